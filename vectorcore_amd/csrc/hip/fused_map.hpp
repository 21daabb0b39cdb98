// Kernels of vc_hip_map (fused elementwise programs), shared by the
// translation units that instantiate them: fused_map_inputs.hip is compiled
// once per input count (VC_MAP_NIN = 1..8) so that the unrolled
// interpreters compile in parallel; fused_map.hip holds the C ABI.
#pragma once

#include "functions.hpp"
#include "reduce_common.hpp"
#include "vc_hip_internal.hpp"

#include <algorithm>

namespace vchip {
namespace fmap {

typedef float f4 __attribute__((ext_vector_type(4)));
// 16 bytes on any 4-byte boundary (a 16-byte load or store needs no more).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kSlots = VC_HIP_MAP_SLOTS;
constexpr int kCode = VC_HIP_MAP_CODE;
constexpr int kShortCode = 16;
constexpr int kInputs = VC_HIP_MAP_INPUTS;
constexpr int kOutputs = VC_HIP_MAP_OUTPUTS;
constexpr int kSums = VC_HIP_MAP_SUMS;
constexpr int kConsts = VC_HIP_MAP_CONSTANTS;
constexpr unsigned kMapBlock = 256;
static_assert(kSlots == 16, "a slot is one element of a 16-wide register vector");

struct Program {
    const float* in[kInputs];
    float* out[kOutputs];
    float* sum[kSums];  // row sums (map_rows_kernel)
    float konst[kConsts];
    uint32_t code[kCode];  // op | a << 8 | b << 16 | dst << 24
    int n_code, n_const, n_out, n_sum;
    uint8_t out_slot[kOutputs];
    uint8_t sum_slot[kSums];
    // Matrix programs (vc_hip_map_broadcast): how each input is indexed
    // (VC_MAP_FULL ...), and the matrix.
    uint8_t kind[kInputs];
    uint32_t extent[kInputs];  // values of an input that is not full
    uint32_t cols, len, count;
    uint32_t cols_magic, cols_shift, len_magic, len_shift;  // for divide()
};

// n / d for n < 2^31 as a multiplication: magic = floor(2^(31 + l) / d) + 1 and
// shift = 31 + l with l = ceil(log2 d) (the error of magic / 2^shift is below
// 2^-shift <= 2^-31 / d, less than what separates n / d from the next whole number).
inline void set_magic(uint32_t d, uint32_t& magic, uint32_t& shift) {
    uint32_t l = 0;
    while ((uint64_t(1) << l) < d) ++l;
    magic = uint32_t((uint64_t(1) << (31 + l)) / d + 1);
    shift = 31 + l;
}
__device__ inline uint32_t divide(uint32_t n, uint32_t magic, uint32_t shift) {
    return uint32_t((uint64_t(n) * magic) >> shift);
}

// The matrix coordinates of a thread's W values: row (group of rows and row in
// the group) and column of each, and whether they lie in one row.
template <int W>
struct Place {
    uint32_t r[W], group[W], in_group[W], c[W];
    bool one_row;
    // Columns c0 .. c0 + W - 1 of row r0, running on into the next rows.
    __device__ void set(const Program& P, uint32_t r0, uint32_t c0) {
        one_row = c0 + W <= P.cols;
        uint32_t g0 = r0, a0 = 0;
        if (P.len != 1) g0 = divide(r0, P.len_magic, P.len_shift), a0 = r0 - g0 * P.len;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            r[j] = r0, group[j] = g0, in_group[j] = a0, c[j] = c0;
            if (++c0 == P.cols) {
                c0 = 0, ++r0;
                if (++a0 == P.len) a0 = 0, ++g0;
            }
        }
    }
};
template <int W>
__device__ inline Place<W> place_of(const Program& P, uint32_t e) {  // elements e .. e + W - 1
    Place<W> at;
    const uint32_t r = divide(e, P.cols_magic, P.cols_shift);
    at.set(P, r, e - r * P.cols);
    return at;
}
template <int W>
__device__ inline Place<W> place_at(const Program& P, uint32_t r, uint32_t c) {
    Place<W> at;
    at.set(P, r, c);
    return at;
}

// W values per slot: one element (W = 1) or four consecutive ones (W = 4).
template <int W>
struct Regs {
    f16v c[W];
};
template <int W>
struct Vals {
    float v[W];
};

template <int W>
__device__ inline Vals<W> get(const Regs<W>& r, int slot) {
    Vals<W> o;
#pragma unroll
    for (int j = 0; j < W; ++j) o.v[j] = r.c[j][slot];
    return o;
}
template <int W>
__device__ inline void put(Regs<W>& r, int slot, const Vals<W>& v) {
#pragma unroll
    for (int j = 0; j < W; ++j) r.c[j][slot] = v.v[j];
}

template <int W>
__device__ inline Vals<W> load(const float* __restrict__ p) {
    Vals<W> o;
    if constexpr (W == 4) {
        const f4 x = __builtin_nontemporal_load(reinterpret_cast<const f4u*>(p));
        o.v[0] = x.x;
        o.v[1] = x.y;
        o.v[2] = x.z;
        o.v[3] = x.w;
    } else {
        o.v[0] = __builtin_nontemporal_load(p);
    }
    return o;
}
template <int W>
__device__ inline void store_any(float* __restrict__ p, const Vals<W>& v) {
    if constexpr (W == 4) *reinterpret_cast<f4u*>(p) = f4{v.v[0], v.v[1], v.v[2], v.v[3]};
    else p[0] = v.v[0];
}
template <int W>
__device__ inline void store(float* __restrict__ p, const Vals<W>& v) {
    if constexpr (W == 4) {
        __builtin_nontemporal_store(f4u{v.v[0], v.v[1], v.v[2], v.v[3]}, reinterpret_cast<f4u*>(p));
    } else {
        __builtin_nontemporal_store(v.v[0], p);
    }
}

// W consecutive values on any 4-byte boundary, through the caches (vectors
// that every row reads).
template <int W>
__device__ inline Vals<W> load_any(const float* __restrict__ p) {
    Vals<W> o;
    if constexpr (W == 4) {
        const f4 x = *reinterpret_cast<const f4u*>(p);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.v[j] = x[j];
    } else {
        o.v[0] = p[0];
    }
    return o;
}

// One instruction on the W values of every slot, for programs whose words are
// unrolled into scalars: what a word decides has to stay in scalar registers
// from one element to the next, so nothing but its operation and slots is
// derived from it. (matrix_step's order and signs spilled 193 scalar registers
// to vector lanes here, 35 this way: two inputs and 20 instructions on 4096 x
// 4096 88 us against 72.)
template <int W>
__device__ inline void plain_step(Regs<W>& r, uint32_t word) {
    const int op = int(word & 255u), ia = int((word >> 8) & 255u), ib = int((word >> 16) & 255u), id = int(word >> 24);
    const Vals<W> a = get(r, ia), b = get(r, ib);
    Vals<W> v;
    switch (op) {
        case VC_MAP_ADD:
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] + b.v[j];
            break;
        case VC_MAP_SUB:
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] - b.v[j];
            break;
        case VC_MAP_MUL:
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] * b.v[j];
            break;
        case VC_MAP_DIV:
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] / b.v[j];
            break;
        case VC_MAP_NEG:
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = -a.v[j];
            break;
        default:  // VC_MAP_STEP
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] > 0.0f ? 1.0f : 0.0f;
            break;
    }
    put(r, id, v);
}

// As plain_step for matrix programs. `at`: the coordinates of the W values.
template <int W>
__device__ inline void matrix_step(Regs<W>& r, const Program& P, const Place<W>& at, uint32_t word) {
    const int op = int(word & 255u), ia = int((word >> 8) & 255u), ib = int((word >> 16) & 255u), id = int(word >> 24);
    const Vals<W> a = get(r, ia);
    Vals<W> v;
    // The commonest operations take the fewest branches (map_columns_kernel<3, 4>, 16 instructions on 4096 x 4096:
    // 90.9 -> 87.6 us; marks that keep a result in registers for the next instruction, at two more branches, took
    // 99, and loading the next row's inputs before the program 90). A subtraction adds the negated operand, the
    // same bits.
    if (op <= VC_MAP_MUL) {
        const Vals<W> b = get(r, ib);
        if (op == VC_MAP_MUL) {
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] * b.v[j];
        } else {  // VC_MAP_ADD or VC_MAP_SUB
            const uint32_t sign = uint32_t(op) << 31;
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] + __uint_as_float(__float_as_uint(b.v[j]) ^ sign);
        }
    } else if (op <= VC_MAP_STEP) {
        if (op == VC_MAP_DIV) {
            const Vals<W> b = get(r, ib);
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = a.v[j] / b.v[j];
        } else {  // VC_MAP_NEG or VC_MAP_STEP
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = op == VC_MAP_NEG ? -a.v[j] : a.v[j] > 0.0f ? 1.0f : 0.0f;
        }
    } else if (op <= VC_MAP_AT_COLUMN) {
        const Vals<W> b = get(r, ib);
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const uint32_t axis = op == VC_MAP_AT_ROW ? at.in_group[j] : at.c[j];
            const uint32_t keep = int(a.v[j]) == int(axis) ? ~0u : 0u;
            v.v[j] = __uint_as_float(__float_as_uint(b.v[j]) & keep);
        }
    } else if (op == VC_MAP_RELU) {
#pragma unroll
        for (int j = 0; j < W; ++j) v.v[j] = ReluOp()(a.v[j]);
    } else if (op == VC_MAP_LOG) {
#pragma unroll
        for (int j = 0; j < W; ++j) v.v[j] = LogOp()(a.v[j]);
    } else {  // VC_MAP_SIGMOID or VC_MAP_EXP, on one exponential
        const bool sigmoid = op == VC_MAP_SIGMOID;
#pragma unroll
        for (int j = 0; j < W; ++j) v.v[j] = ExpOp()(sigmoid ? -fabsf(a.v[j]) : a.v[j]);
        if (sigmoid)
#pragma unroll
            for (int j = 0; j < W; ++j) v.v[j] = SigmoidOp::of(a.v[j], v.v[j]);
    }
    put(r, id, v);
}

// The program. Its words are kernel arguments: flat and plain column programs
// unroll the first Code of them (Code >= n_code), so that every word is a
// scalar. Matrix programs, whose functions make an instruction's code long, loop
// over one copy of it, each word loaded while the one before runs: the unrolled
// copies are no faster (bias, activations and their product on 4096 x 4096 with
// gradients, 16 instructions: 116-127 us, 119 looped; rows of 8192 x 1024 to
// mean 0 and variance 1: 229 us, 224 looped), and eight times the code.
template <int Code, bool Matrix, int W>
__device__ inline void run(Regs<W>& r, const Program& P, const Place<W>& at, uint32_t words = 0) {
    if constexpr (Matrix) {
#pragma nounroll
        for (int k = 0; k < P.n_code; ++k)
            matrix_step(r, P, at, uint32_t(__builtin_amdgcn_readlane(int(words), k)));
    } else {
#pragma unroll
        for (int k = 0; k < Code; ++k) {
            if (k >= P.n_code) continue;  // uniform: the rest of the loop is skipped
            plain_step(r, P.code[k]);
        }
    }
}

template <int W>
__device__ inline void set_constants(Regs<W>& r, const Program& P, int n_in) {
#pragma nounroll
    for (int c = 0; c < P.n_const; ++c) {
        Vals<W> v;
#pragma unroll
        for (int j = 0; j < W; ++j) v.v[j] = P.konst[c];
        put(r, n_in + c, v);
    }
}

// Loads element group e (W consecutive values) of every input into its slot.
// (Loading the next group ahead of the computation measured no faster: the
// other waves of the CU hide the latency.)
template <int NIn, int W>
__device__ inline void load_inputs(Regs<W>& r, const Program& P, int64_t e) {
    Vals<W> v[NIn];
#pragma unroll
    for (int j = 0; j < NIn; ++j) v[j] = load<W>(P.in[j] + e);
#pragma unroll
    for (int j = 0; j < NIn; ++j) put(r, j, v[j]);
}

// As load_inputs for a matrix program: element group e lies at `at`.
template <int NIn, int W>
__device__ inline void load_matrix_inputs(Regs<W>& r, const Program& P, int64_t e, const Place<W>& at) {
    Vals<W> v[NIn];
#pragma unroll
    for (int j = 0; j < NIn; ++j) {
        const float* in = P.in[j];
        if (P.kind[j] == VC_MAP_FULL) {
            v[j] = load_any<W>(in + e);
        } else if (P.kind[j] == VC_MAP_PER_COLUMN) {
            if (at.one_row) v[j] = load_any<W>(in + at.c[0]);
            else
#pragma unroll
                for (int w = 0; w < W; ++w) v[j].v[w] = in[at.c[w]];
        } else if (P.kind[j] == VC_MAP_PER_ROW) {
            v[j].v[0] = in[at.r[0]];
#pragma unroll
            for (int w = 1; w < W; ++w) v[j].v[w] = at.one_row ? v[j].v[0] : in[at.r[w]];
        } else {  // VC_MAP_PER_GROUP
            if (at.one_row) v[j] = load_any<W>(in + int64_t(at.group[0]) * P.cols + at.c[0]);
            else
#pragma unroll
                for (int w = 0; w < W; ++w) v[j].v[w] = in[int64_t(at.group[w]) * P.cols + at.c[w]];
        }
    }
#pragma unroll
    for (int j = 0; j < NIn; ++j) put(r, j, v[j]);
}

// As load_matrix_inputs where every lane's values lie in one row: each input is
// one buffer load of W values whatever its kind, so that all of them are in
// flight together (with a branch per kind each load was waited for before the
// next: bias, activations and their product on 4096 x 4096 with gradients 123 us, 94 now). Element e_base (the same in all
// lanes) + e_off is the lane's first; a one-value-per-row input's load starts
// with its value and may run past the input, where the descriptor ends it.
// Lane offsets fit 32 bits: e_off is below 2^28, and an input that is not
// full has fewer than 2^30 values (see vc_hip_map_broadcast).
template <int NIn, int W>
__device__ inline void load_row_inputs(Regs<W>& r, const Program& P, uint32_t e_base, uint32_t e_off, const Place<W>& at) {
    Vals<W> v[NIn];
    const uint32_t in_group = at.group[0] * P.cols + at.c[0];
#pragma unroll
    for (int j = 0; j < NIn; ++j) {
        const int kind = P.kind[j];
        const bool full = kind == VC_MAP_FULL;
        const uint32_t rest = P.count - e_base;
        const uint32_t extent = full ? (rest < (1u << 29) ? rest : (1u << 29)) : P.extent[j];
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(P.in[j] + (full ? e_base : 0u)), short(0), int(extent * 4u), 0x00020000);
        const uint32_t at_j = full ? e_off : kind == VC_MAP_PER_COLUMN ? at.c[0] : kind == VC_MAP_PER_ROW ? at.r[0] : in_group;
        if constexpr (W == 4) {
            const f4 x = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, at_j * 4u, 0, 0));
#pragma unroll
            for (int w = 0; w < 4; ++w) v[j].v[w] = x[w];
        } else {
            v[j].v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at_j * 4u, 0, 0));
        }
    }
#pragma unroll
    for (int j = 0; j < NIn; ++j) {
#pragma unroll
        for (int w = 1; w < W; ++w) v[j].v[w] = P.kind[j] == VC_MAP_PER_ROW ? v[j].v[0] : v[j].v[w];
        put(r, j, v[j]);
    }
}

// Lane k holds instruction k of a matrix program: a readlane gives a word as a
// scalar, without a wait on the scalar cache for each.
__device__ inline uint32_t lane_words(const Program& P) {
    static_assert(kCode <= 64, "a wavefront holds a program");
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t word = P.code[lane < uint32_t(kCode) ? lane : 0u];
    asm volatile("" : "+v"(word));  // loaded here, in every lane, not in a branch that some lanes do not take
    return word;
}

template <int W>
__device__ inline void store_outputs(const Regs<W>& r, const Program& P, int64_t e) {
#pragma unroll
    for (int j = 0; j < kOutputs; ++j)
        if (j < P.n_out) store<W>(P.out[j] + e, get(r, P.out_slot[j]));
}

// The first element of group g: the last group of a count that is no multiple
// of W ends with the count, and computes and writes what it shares with the group
// before it once more (the same values). A launch of its own for these elements
// cost 2.5 us and the host's part.
template <int W>
__device__ inline int64_t group_start(int64_t g, int64_t count) {
    return W == 1 || g * W < count - W ? g * W : count - W;
}

// Elements [0, count) (count >= W) in groups of W: thread t takes groups t, t + threads, ...
template <int NIn, int W, int Code>
__global__ __launch_bounds__(kMapBlock) void map_flat_kernel(Program P, int64_t count) {
    Regs<W> r;
    set_constants(r, P, NIn);
    const int64_t stride = int64_t(gridDim.x) * blockDim.x, groups = (count + W - 1) / W;
    for (int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < groups; g += stride) {
        const int64_t e = group_start<W>(g, count);
        load_inputs<NIn, W>(r, P, e);
        run<Code, false>(r, P, Place<W>{});
        store_outputs(r, P, e);
    }
}

// map_flat_kernel of a matrix program: full inputs and outputs are read and
// written as there, whatever the columns; the other inputs by coordinates.
// OneRow: W values never cross the end of a row (W = 1, or cols % 4 == 0).
template <int NIn, int W, bool OneRow>
__global__ __launch_bounds__(kMapBlock) void map_matrix_kernel(Program P, int64_t count) {
    Regs<W> r;
    set_constants(r, P, NIn);
    const uint32_t words = lane_words(P);
    const int64_t stride = int64_t(gridDim.x) * blockDim.x, groups = (count + W - 1) / W;
    for (int64_t g0 = int64_t(blockIdx.x) * blockDim.x; g0 < groups; g0 += stride) {
        const int64_t g = g0 + threadIdx.x;
        if (g >= groups) break;
        const int64_t e = group_start<W>(g, count);
        const Place<W> at = place_of<W>(P, uint32_t(e));
        if constexpr (OneRow) load_row_inputs<NIn, W>(r, P, uint32_t(g0 * W), threadIdx.x * W, at);
        else load_matrix_inputs<NIn, W>(r, P, e, at);
        run<0, true>(r, P, at, words);
        store_outputs(r, P, e);
    }
}

// A matrix program with the row sums of P.sum_slot[s] for s < P.n_sum: Lanes
// threads (a wavefront or the workgroup) take a row, W columns at a time; the
// last group of a row whose length is no multiple of W is moved back to end
// with the row (its first values are computed and written twice, and added
// once). Sums in double: each lane in column order, then red::wave_sum's order,
// then wave order.
template <int NIn, int W, int Lanes>
__global__ __launch_bounds__(kMapBlock) void map_rows_kernel(Program P, int64_t rows) {
    constexpr int kWaves = Lanes / 64;
    __shared__ double wave_part[kSums][4];
    const int t = int(threadIdx.x) % Lanes, lane = int(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const uint32_t cols = P.cols;
    Regs<W> r;
    set_constants(r, P, NIn);
    const uint32_t words = lane_words(P);
    const int64_t step = int64_t(gridDim.x) * (kMapBlock / Lanes);
    for (int64_t row = int64_t(blockIdx.x) * (kMapBlock / Lanes) + wave / kWaves; row < rows; row += step) {
        double acc[kSums] = {0.0, 0.0};
        for (uint32_t c0 = 0; c0 < cols; c0 += Lanes * W) {
            const uint32_t c = c0 + uint32_t(t) * W;
            if (c >= cols) break;
            const uint32_t c1 = c + W <= cols ? c : cols - W;
            const uint32_t before = c0 < W ? c0 : W;  // c1 may lie in the group before c0
            const int64_t e = row * cols + c1;
            const Place<W> at = place_at<W>(P, uint32_t(row), c1);
            load_row_inputs<NIn, W>(r, P, uint32_t(row) * cols + (c0 - before), c1 - (c0 - before), at);
            run<0, true>(r, P, at, words);
#pragma unroll
            for (int j = 0; j < kOutputs; ++j)
                if (j < P.n_out) store_any<W>(P.out[j] + e, get(r, P.out_slot[j]));
#pragma unroll
            for (int s = 0; s < kSums; ++s)
                if (s < P.n_sum) {
                    const Vals<W> v = get(r, P.sum_slot[s]);
#pragma unroll
                    for (int j = 0; j < W; ++j) acc[s] += c1 + uint32_t(j) >= c ? double(v.v[j]) : 0.0;
                }
        }
#pragma unroll
        for (int s = 0; s < kSums; ++s) acc[s] = red::wave_sum(acc[s]);
        if constexpr (kWaves > 1) {
            if (lane == 0)
                for (int s = 0; s < kSums; ++s) wave_part[s][wave] = acc[s];
            __syncthreads();
            for (int s = 0; s < kSums; ++s) {
                acc[s] = wave_part[s][0];
                for (int k = 1; k < kWaves; ++k) acc[s] += wave_part[s][k];
            }
            __syncthreads();
        }
        if (t == 0)
            for (int s = 0; s < P.n_sum; ++s) P.sum[s][row] = float(acc[s]);
    }
}

// A [rows, cols] view, with the column sums of P.sum_slot[s] for s < NSum.
// Workgroup (x, y) of a grid (col_blocks, gy) takes columns
// [x * 64 W, (x + 1) * 64 W): lane l holds W consecutive columns, and wave w
// the rows w + 4 y, w + 4 y + 4 gy, w + 4 y + 8 gy, ... (at any moment the
// grid streams a contiguous band of rows). Each lane adds its values in double
// in row order; the four waves' sums are added in wave order and written as
// partial row y: part[s][y][col]. column_partials_kernel then adds the gy
// partial rows in a fixed order.
template <int NIn, int W, int Code, int NSum, bool Matrix>
__global__ __launch_bounds__(kMapBlock) void map_columns_kernel(Program P, int64_t rows, int64_t cols,
                                                                double* __restrict__ part) {
    __shared__ double wave_part[NSum][4][64 * W];
    const int lane = int(threadIdx.x) & 63;
    const int w = Matrix ? __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6) : int(threadIdx.x) >> 6;
    const int64_t col = (int64_t(blockIdx.x) * 64 + lane) * W;
    const uint32_t words = Matrix ? lane_words(P) : 0;
    const int64_t step = 4 * int64_t(gridDim.y);
    Regs<W> r;
    set_constants(r, P, NIn);
    double acc[NSum][W];
#pragma unroll
    for (int s = 0; s < NSum; ++s)
#pragma unroll
        for (int j = 0; j < W; ++j) acc[s][j] = 0.0;
    if (col < cols) {
        for (int64_t row = int64_t(blockIdx.y) * 4 + w; row < rows; row += step) {
            const int64_t e = row * cols + col;
            if constexpr (Matrix) {
                const Place<W> at = place_at<W>(P, uint32_t(row), uint32_t(col));
                load_row_inputs<NIn, W>(r, P, uint32_t(row) * uint32_t(cols) + blockIdx.x * 64 * W, uint32_t(lane) * W, at);
                run<Code, true>(r, P, at, words);
            } else {
                load_inputs<NIn, W>(r, P, e);
                run<Code, false>(r, P, Place<W>{});
            }
            store_outputs(r, P, e);
#pragma unroll
            for (int s = 0; s < NSum; ++s) {
                if (s < P.n_sum) {
                    const Vals<W> v = get(r, P.sum_slot[s]);
#pragma unroll
                    for (int j = 0; j < W; ++j) acc[s][j] += double(v.v[j]);
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NSum; ++s)
#pragma unroll
        for (int j = 0; j < W; ++j) wave_part[s][w][lane * W + j] = acc[s][j];
    __syncthreads();
    if (w == 0 && col < cols) {
        for (int s = 0; s < P.n_sum; ++s) {
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const int i = lane * W + j;
                const double t = ((wave_part[s][0][i] + wave_part[s][1][i]) + wave_part[s][2][i]) + wave_part[s][3][i];
                if (col + j < cols) part[(int64_t(s) * gridDim.y + blockIdx.y) * cols + col + j] = t;
            }
        }
    }
}

// Flat launches: at most 4096 workgroups (16 per CU), each thread looping.
constexpr unsigned kFlatBlocks = 4096;

template <int NIn>
void launch_flat(Device& d, const Program& P, int64_t count, bool vec) {
    vec = vec && count >= 4;
    const dim3 grid(grid_1d(size_t(vec ? (count + 3) / 4 : count), kMapBlock, kFlatBlocks));
    if (!vec) launch(map_flat_kernel<NIn, 1, kCode>, grid, dim3(kMapBlock), 0, d.stream, P, count);
    else if (P.n_code <= kShortCode) launch(map_flat_kernel<NIn, 4, kShortCode>, grid, dim3(kMapBlock), 0, d.stream, P, count);
    else launch(map_flat_kernel<NIn, 4, kCode>, grid, dim3(kMapBlock), 0, d.stream, P, count);
}

// The column traversal's grid: about 2048 workgroups, with gy (the number of
// partial rows) at most rows / 4. A function of the shape only, so the order
// of every column sum is too.
struct ColumnGrid {
    int64_t col_blocks, gy;
};
inline ColumnGrid column_grid(int64_t rows, int64_t cols, int w) {
    ColumnGrid g{};
    g.col_blocks = (cols + 64 * w - 1) / (64 * w);
    g.gy = (2048 + g.col_blocks - 1) / g.col_blocks;
    const int64_t max_gy = (rows + 3) / 4;
    if (g.gy > max_gy) g.gy = max_gy;
    if (g.gy < 1) g.gy = 1;
    return g;
}

template <int NIn>
void launch_columns(Device& d, const Program& P, int64_t rows, int64_t cols, bool vec, double* part) {
    const ColumnGrid g = column_grid(rows, cols, vec ? 4 : 1);
    const dim3 grid(unsigned(g.col_blocks), unsigned(g.gy));
    if (P.cols != 0) {  // a matrix program
        if (vec && P.n_sum == 1)
            launch(map_columns_kernel<NIn, 4, kCode, 1, true>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
        else if (vec)
            launch(map_columns_kernel<NIn, 4, kCode, kSums, true>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
        else
            launch(map_columns_kernel<NIn, 1, kCode, kSums, true>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
    } else if (vec && P.n_code <= kShortCode && P.n_sum == 1) {  // the common case: a short program, one sum
        launch(map_columns_kernel<NIn, 4, kShortCode, 1, false>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
    } else if (vec) {
        launch(map_columns_kernel<NIn, 4, kCode, kSums, false>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
    } else {
        launch(map_columns_kernel<NIn, 1, kCode, kSums, false>, grid, dim3(kMapBlock), 0, d.stream, P, rows, cols, part);
    }
}

// A matrix program without sums.
template <int NIn>
void launch_matrix(Device& d, const Program& P, int64_t count, bool vec) {
    vec = vec && count >= 4;
    const dim3 grid(grid_1d(size_t(vec ? (count + 3) / 4 : count), kMapBlock, kFlatBlocks));
    if (!vec) launch(map_matrix_kernel<NIn, 1, true>, grid, dim3(kMapBlock), 0, d.stream, P, count);
    else if (P.cols % 4 == 0) launch(map_matrix_kernel<NIn, 4, true>, grid, dim3(kMapBlock), 0, d.stream, P, count);
    else launch(map_matrix_kernel<NIn, 4, false>, grid, dim3(kMapBlock), 0, d.stream, P, count);
}

// A matrix program with row sums: a wavefront per row, or a workgroup for few long rows.
template <int NIn>
void launch_rows(Device& d, const Program& P, int64_t rows) {
    const bool wide = rows < 2048 && P.cols > 1024;
    const unsigned grid = unsigned(std::min<int64_t>(wide ? rows : (rows + 3) / 4, kFlatBlocks));
    if (P.cols < 4) launch(map_rows_kernel<NIn, 1, 64>, dim3(grid), dim3(kMapBlock), 0, d.stream, P, rows);
    else if (wide) launch(map_rows_kernel<NIn, 4, 256>, dim3(grid), dim3(kMapBlock), 0, d.stream, P, rows);
    else launch(map_rows_kernel<NIn, 4, 64>, dim3(grid), dim3(kMapBlock), 0, d.stream, P, rows);
}

}  // namespace fmap
}  // namespace vchip
