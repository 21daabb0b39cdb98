// Softmax and log-softmax along one axis of [outer, length, inner], and their
// gradients, in one pass each: the composition of src/ops.cpp:416-424
// (x - max, exp, sum, log, subtract, exp) and of its backward rules, with the
// same fp32 operations per element and sums accumulated in double, in a fixed
// order.
//
// Bound by HBM: the forward reads x and writes the result, the backward reads
// the upstream gradient and x (the values in between are computed again from
// the row's maximum and sum) and writes the gradient. Composed, the two
// directions were eleven passes over memory: 6000 x 1003 forward and backward
// 128 us, now 23.
#include "reduce_common.hpp"
#include "vc_hip_internal.hpp"

#include <algorithm>
#include <string>

namespace vchip {
namespace {

using red::kWave;

constexpr int kRowBlock = 256;

typedef float f4 __attribute__((ext_vector_type(4)));
// 16 bytes on any 4-byte boundary, as rows of any length start.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// Maximum by the reference's scan from element 0 with strict '>'
// (src/cpu/cpu_backend.cpp:443-457): NaN never wins, but a NaN first element
// stays (the caller's check).
__device__ inline float wave_max(float m) {
    const int lane = red::lane_id();
    const auto larger = [](float a, float b) { return b > a ? b : a; };
    m = larger(m, red::partner<0>(m, lane));
    m = larger(m, red::partner<1>(m, lane));
    m = larger(m, red::partner<2>(m, lane));
    m = larger(m, red::partner<3>(m, lane));
    m = larger(m, red::partner<4>(m, lane));
    m = larger(m, red::partner<5>(m, lane));
    return m;
}

constexpr float kLowest = -__builtin_huge_valf();

// What one element contributes, from x and its row's maximum, sum and the sum's logarithm.
template <bool Log>
__device__ inline float result(float x, float m, float l) {
    const float y = (x - m) - l;
    return Log ? y : expf(y);
}
// The gradient that reaches log_softmax's rule: softmax is its exp.
template <bool Log>
__device__ inline float through_exp(float g, float x, float m, float l) {
    return Log ? g : g * result<false>(x, m, l);
}

// NV groups of four consecutive values per lane: row values 4 lane + 256 u ..
template <int NV>
__device__ inline void load_row(const float* __restrict__ row, int len, int lane, float fill, f4 (&v)[NV]) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int a = 4 * lane + 256 * u;
        if (a + 3 < len) {
            v[u] = *reinterpret_cast<const f4u*>(row + a);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[u][e] = a + e < len ? row[a + e] : fill;
        }
    }
}
template <int NV>
__device__ inline void store_row(float* __restrict__ row, int len, int lane, const f4 (&v)[NV]) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int a = 4 * lane + 256 * u;
        if (a + 3 < len) {
            *reinterpret_cast<f4u*>(row + a) = v[u];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (a + e < len) row[a + e] = v[u][e];
        }
    }
}

// Rows of up to 256 NV values: a wavefront per row, the row in registers.
template <bool Log, int NV>
__global__ __launch_bounds__(kRowBlock) void rows_forward_kernel(const float* __restrict__ x, float* __restrict__ y,
                                                                 float* __restrict__ stats, int64_t rows, int len) {
    const int lane = threadIdx.x % kWave;
    const int64_t step = int64_t(gridDim.x) * (kRowBlock / kWave);
    for (int64_t r = int64_t(blockIdx.x) * (kRowBlock / kWave) + threadIdx.x / kWave; r < rows; r += step) {
        f4 v[NV];
        load_row(x + r * len, len, lane, kLowest, v);
        float m = kLowest;
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = v[u][e] > m ? v[u][e] : m;
        m = wave_max(m);
        const float first = __shfl(v[0][0], 0, kWave);
        if (first != first) m = first;
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * lane + 256 * u + e < len) sum += double(expf(v[u][e] - m));
        const float s = float(red::wave_sum(sum));
        const float l = logf(s);
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[u][e] = result<Log>(v[u][e], m, l);
        store_row(y + r * len, len, lane, v);
        if (stats && lane == 0) {
            stats[2 * r] = m;
            stats[2 * r + 1] = s;
        }
    }
}

template <bool Log, int NV>
__global__ __launch_bounds__(kRowBlock) void rows_backward_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                                  const float* __restrict__ stats, float* __restrict__ dx,
                                                                  int64_t rows, int len) {
    const int lane = threadIdx.x % kWave;
    const int64_t step = int64_t(gridDim.x) * (kRowBlock / kWave);
    for (int64_t r = int64_t(blockIdx.x) * (kRowBlock / kWave) + threadIdx.x / kWave; r < rows; r += step) {
        f4 v[NV], w[NV];
        load_row(x + r * len, len, lane, 0.0f, v);
        load_row(g + r * len, len, lane, 0.0f, w);
        const float m = stats[2 * r], s = stats[2 * r + 1], l = logf(s);
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                w[u][e] = through_exp<Log>(w[u][e], v[u][e], m, l);
                if (4 * lane + 256 * u + e < len) sum += double(w[u][e]);
            }
        const float ds = -float(red::wave_sum(sum)) / s + 0.0f;
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) w[u][e] = w[u][e] + ds * expf(v[u][e] - m);
        store_row(dx + r * len, len, lane, w);
    }
}

// Longer rows: a workgroup per row, which the caches hold between its passes.
constexpr int kLongBlock = 512;

template <bool Log>
__global__ __launch_bounds__(kLongBlock) void long_forward_kernel(const float* __restrict__ x, float* __restrict__ y,
                                                                  float* __restrict__ stats, int64_t rows, int64_t len) {
    __shared__ float part_max[kLongBlock / kWave];
    __shared__ double part_sum[kLongBlock / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float* row = x + r * len;
        float m = kLowest;
        for (int64_t a = threadIdx.x; a < len; a += kLongBlock) m = row[a] > m ? row[a] : m;
        m = wave_max(m);
        if (lane == 0) part_max[wave] = m;
        __syncthreads();
        for (int k = 0; k < kLongBlock / kWave; ++k) m = part_max[k] > m ? part_max[k] : m;
        const float first = row[0];
        if (first != first) m = first;
        double sum = 0.0;
        for (int64_t a = threadIdx.x; a < len; a += kLongBlock) sum += double(expf(row[a] - m));
        sum = red::wave_sum(sum);
        if (lane == 0) part_sum[wave] = sum;
        __syncthreads();
        sum = part_sum[0];
        for (int k = 1; k < kLongBlock / kWave; ++k) sum += part_sum[k];
        const float s = float(sum), l = logf(s);
        for (int64_t a = threadIdx.x; a < len; a += kLongBlock) y[r * len + a] = result<Log>(row[a], m, l);
        if (stats && threadIdx.x == 0) {
            stats[2 * r] = m;
            stats[2 * r + 1] = s;
        }
        __syncthreads();
    }
}

template <bool Log>
__global__ __launch_bounds__(kLongBlock) void long_backward_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                                   const float* __restrict__ stats, float* __restrict__ dx,
                                                                   int64_t rows, int64_t len) {
    __shared__ double part_sum[kLongBlock / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float *gr = g + r * len, *row = x + r * len;
        const float m = stats[2 * r], s = stats[2 * r + 1], l = logf(s);
        double sum = 0.0;
        for (int64_t a = threadIdx.x; a < len; a += kLongBlock) sum += double(through_exp<Log>(gr[a], row[a], m, l));
        sum = red::wave_sum(sum);
        if (lane == 0) part_sum[wave] = sum;
        __syncthreads();
        sum = part_sum[0];
        for (int k = 1; k < kLongBlock / kWave; ++k) sum += part_sum[k];
        const float ds = -float(sum) / s + 0.0f;
        for (int64_t a = threadIdx.x; a < len; a += kLongBlock)
            dx[r * len + a] = through_exp<Log>(gr[a], row[a], m, l) + ds * expf(row[a] - m);
        __syncthreads();
    }
}

// inner > 1: a workgroup takes 16 adjacent columns of one outer index, its 32
// row lanes walk the axis with eight rows in flight, and their partial results
// are joined through LDS in lane order.
constexpr int kCols = 16, kRowLanes = 32;

// f(a, values) for the rows a of this lane, in order, x[a] loaded eight rows ahead.
template <class F>
__device__ inline void walk(const float* __restrict__ x, int64_t len, int64_t inner, int rl, bool inside, F f) {
    if (!inside) return;
    for (int64_t a0 = rl; a0 < len; a0 += 8 * kRowLanes) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = a0 + u * kRowLanes < len ? x[(a0 + u * kRowLanes) * inner] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (a0 + u * kRowLanes < len) f(a0 + u * kRowLanes, v[u]);
    }
}
template <class F>
__device__ inline void walk2(const float* __restrict__ x, const float* __restrict__ g, int64_t len, int64_t inner, int rl,
                             bool inside, F f) {
    if (!inside) return;
    for (int64_t a0 = rl; a0 < len; a0 += 4 * kRowLanes) {
        float v[4], w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool in = a0 + u * kRowLanes < len;
            v[u] = in ? x[(a0 + u * kRowLanes) * inner] : 0.0f;
            w[u] = in ? g[(a0 + u * kRowLanes) * inner] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (a0 + u * kRowLanes < len) f(a0 + u * kRowLanes, v[u], w[u]);
    }
}

// The sum of the column's row lanes, in lane order; every lane gets it.
__device__ inline double column_total(double v, double (*part)[kCols], int c, int rl) {
    part[rl][c] = v;
    __syncthreads();
    double total = part[0][c];
    for (int k = 1; k < kRowLanes; ++k) total += part[k][c];
    __syncthreads();
    return total;
}

template <bool Log>
__global__ __launch_bounds__(kCols * kRowLanes) void cols_forward_kernel(const float* __restrict__ x, float* __restrict__ y,
                                                                         float* __restrict__ stats, int64_t len,
                                                                         int64_t inner, int64_t blocks_per_outer) {
    __shared__ double part[kRowLanes][kCols];
    const int c = threadIdx.x % kCols, rl = threadIdx.x / kCols;
    const int64_t o = blockIdx.x / blocks_per_outer, col = (blockIdx.x % blocks_per_outer) * kCols + c;
    const bool inside = col < inner;
    const int64_t base = o * len * inner + col;
    float m = kLowest;
    walk(x + base, len, inner, rl, inside, [&](int64_t, float v) { m = v > m ? v : m; });
    part[rl][c] = double(m);
    __syncthreads();
    for (int k = 0; k < kRowLanes; ++k) m = float(part[k][c]) > m ? float(part[k][c]) : m;
    __syncthreads();
    if (inside) {
        const float first = x[base];
        if (first != first) m = first;
    }
    double sum = 0.0;
    walk(x + base, len, inner, rl, inside, [&](int64_t, float v) { sum += double(expf(v - m)); });
    const float s = float(column_total(sum, part, c, rl)), l = logf(s);
    walk(x + base, len, inner, rl, inside, [&](int64_t a, float v) { y[base + a * inner] = result<Log>(v, m, l); });
    if (stats && inside && rl == 0) {
        stats[2 * (o * inner + col)] = m;
        stats[2 * (o * inner + col) + 1] = s;
    }
}

template <bool Log>
__global__ __launch_bounds__(kCols * kRowLanes) void cols_backward_kernel(const float* __restrict__ g,
                                                                          const float* __restrict__ x,
                                                                          const float* __restrict__ stats,
                                                                          float* __restrict__ dx, int64_t len, int64_t inner,
                                                                          int64_t blocks_per_outer) {
    __shared__ double part[kRowLanes][kCols];
    const int c = threadIdx.x % kCols, rl = threadIdx.x / kCols;
    const int64_t o = blockIdx.x / blocks_per_outer, col = (blockIdx.x % blocks_per_outer) * kCols + c;
    const bool inside = col < inner;
    const int64_t base = o * len * inner + col;
    const float m = inside ? stats[2 * (o * inner + col)] : 0.0f, s = inside ? stats[2 * (o * inner + col) + 1] : 1.0f;
    const float l = logf(s);
    double sum = 0.0;
    walk2(x + base, g + base, len, inner, rl, inside,
          [&](int64_t, float v, float w) { sum += double(through_exp<Log>(w, v, m, l)); });
    const float ds = -float(column_total(sum, part, c, rl)) / s + 0.0f;
    walk2(x + base, g + base, len, inner, rl, inside, [&](int64_t a, float v, float w) {
        dx[base + a * inner] = through_exp<Log>(w, v, m, l) + ds * expf(v - m);
    });
}

// inner > 1, many columns of few elements: a thread per column, which walks
// the axis in order (the later walks find it in the caches).
template <bool Log>
__global__ __launch_bounds__(kRowBlock) void thin_forward_kernel(const float* __restrict__ x, float* __restrict__ y,
                                                                 float* __restrict__ stats, int64_t outer, int64_t len,
                                                                 int64_t inner) {
    const int64_t total = outer * inner, stride = int64_t(gridDim.x) * kRowBlock;
    for (int64_t t = int64_t(blockIdx.x) * kRowBlock + threadIdx.x; t < total; t += stride) {
        const int64_t o = t / inner, base = o * len * inner + (t - o * inner);
        float m = x[base];  // a NaN first element stays
#pragma unroll 4
        for (int64_t a = 1; a < len; ++a) m = x[base + a * inner] > m ? x[base + a * inner] : m;
        double sum = 0.0;
#pragma unroll 4
        for (int64_t a = 0; a < len; ++a) sum += double(expf(x[base + a * inner] - m));
        const float s = float(sum), l = logf(s);
#pragma unroll 4
        for (int64_t a = 0; a < len; ++a) y[base + a * inner] = result<Log>(x[base + a * inner], m, l);
        if (stats) {
            stats[2 * t] = m;
            stats[2 * t + 1] = s;
        }
    }
}

template <bool Log>
__global__ __launch_bounds__(kRowBlock) void thin_backward_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                                  const float* __restrict__ stats, float* __restrict__ dx,
                                                                  int64_t outer, int64_t len, int64_t inner) {
    const int64_t total = outer * inner, stride = int64_t(gridDim.x) * kRowBlock;
    for (int64_t t = int64_t(blockIdx.x) * kRowBlock + threadIdx.x; t < total; t += stride) {
        const int64_t o = t / inner, base = o * len * inner + (t - o * inner);
        const float m = stats[2 * t], s = stats[2 * t + 1], l = logf(s);
        double sum = 0.0;
#pragma unroll 4
        for (int64_t a = 0; a < len; ++a) sum += double(through_exp<Log>(g[base + a * inner], x[base + a * inner], m, l));
        const float ds = -float(sum) / s + 0.0f;
#pragma unroll 4
        for (int64_t a = 0; a < len; ++a)
            dx[base + a * inner] = through_exp<Log>(g[base + a * inner], x[base + a * inner], m, l) +
                                   ds * expf(x[base + a * inner] - m);
    }
}

// The launch of a row or column kernel for [outer, len, inner].
template <class Rows, class Long, class Cols, class Thin>
void dispatch(Device& d, int64_t outer, int64_t len, int64_t inner, Rows rows, Long longer, Cols cols, Thin thin) {
    if (inner == 1) {
        const unsigned grid = unsigned(std::min<int64_t>((outer + 3) / 4, int64_t(d.cu_count) * 64));
        const int64_t nv = (len + 255) / 256;
        if (nv <= 1) rows(std::integral_constant<int, 1>{}, grid);
        else if (nv <= 2) rows(std::integral_constant<int, 2>{}, grid);
        else if (nv <= 4) rows(std::integral_constant<int, 4>{}, grid);
        else if (nv <= 8) rows(std::integral_constant<int, 8>{}, grid);
        else longer(unsigned(std::min<int64_t>(outer, int64_t(d.cu_count) * 16)));
        return;
    }
    const int64_t per_outer = (inner + kCols - 1) / kCols, groups = outer * per_outer, total = outer * inner;
    // A workgroup per 16 columns costs about 3 ns per 256 rows once the chip is full, a thread per column 0.1 us per
    // row for as many columns as the chip holds (512 x 128 x 16, both directions: 13 against 67 us; 4096 x 64 x 16: 70
    // against 47; 100000 x 16 x 2: 856 against 80; composed 132). The first is thus chosen for fewer than 8600
    // workgroups only.
    if (0.003 * double(groups) * double((len + 255) / 256) <= 0.1 * double(len) * std::max(1.0, double(total) / 262144.0))
        cols(unsigned(groups), per_outer);
    else
        thin(grid_1d(size_t(total), kRowBlock, unsigned(d.cu_count) * 64));
}

}  // namespace
}  // namespace vchip

using namespace vchip;

extern "C" {

int vc_hip_softmax_forward(const float* in, float* out, float* stats, size_t outer, size_t length, size_t inner,
                           int log_output) {
    return guard([&] {
        Device& d = require_device();
        const int64_t o = int64_t(outer), len = int64_t(length), n = int64_t(inner);
        if (o == 0 || n == 0) return;
        if (len == 0) fail(VC_HIP_ERR_INVALID_ARGUMENT, "softmax over an empty axis is undefined");
        if (!in || !out) fail(VC_HIP_ERR_INVALID_ARGUMENT, "softmax_forward: null buffer");
        Profiled p("softmax_forward", 0.0, 8.0 * double(o * len * n));
        const auto launch_all = [&](auto log_c) {
            constexpr bool Log = decltype(log_c)::value;
            dispatch(
                d, o, len, n,
                [&](auto nv, unsigned grid) {
                    launch(rows_forward_kernel<Log, decltype(nv)::value>, dim3(grid), dim3(kRowBlock), 0, d.stream, in, out,
                           stats, o, int(len));
                },
                [&](unsigned grid) {
                    launch(long_forward_kernel<Log>, dim3(grid), dim3(kLongBlock), 0, d.stream, in, out, stats, o, len);
                },
                [&](unsigned grid, int64_t per_outer) {
                    launch(cols_forward_kernel<Log>, dim3(grid), dim3(kCols * kRowLanes), 0, d.stream, in, out, stats, len,
                           n, per_outer);
                },
                [&](unsigned grid) {
                    launch(thin_forward_kernel<Log>, dim3(grid), dim3(kRowBlock), 0, d.stream, in, out, stats, o, len, n);
                });
        };
        if (log_output) launch_all(std::true_type{});
        else launch_all(std::false_type{});
        after_launch("softmax_forward");
        p.done();
    });
}

int vc_hip_softmax_backward(const float* grad, const float* in, const float* stats, float* out, size_t outer,
                            size_t length, size_t inner, int log_output) {
    return guard([&] {
        Device& d = require_device();
        const int64_t o = int64_t(outer), len = int64_t(length), n = int64_t(inner);
        if (o * len * n == 0) return;
        if (!grad || !in || !stats || !out) fail(VC_HIP_ERR_INVALID_ARGUMENT, "softmax_backward: null buffer");
        Profiled p("softmax_backward", 0.0, 12.0 * double(o * len * n));
        const auto launch_all = [&](auto log_c) {
            constexpr bool Log = decltype(log_c)::value;
            dispatch(
                d, o, len, n,
                [&](auto nv, unsigned grid) {
                    launch(rows_backward_kernel<Log, decltype(nv)::value>, dim3(grid), dim3(kRowBlock), 0, d.stream, grad,
                           in, stats, out, o, int(len));
                },
                [&](unsigned grid) {
                    launch(long_backward_kernel<Log>, dim3(grid), dim3(kLongBlock), 0, d.stream, grad, in, stats, out, o,
                           len);
                },
                [&](unsigned grid, int64_t per_outer) {
                    launch(cols_backward_kernel<Log>, dim3(grid), dim3(kCols * kRowLanes), 0, d.stream, grad, in, stats,
                           out, len, n, per_outer);
                },
                [&](unsigned grid) {
                    launch(thin_backward_kernel<Log>, dim3(grid), dim3(kRowBlock), 0, d.stream, grad, in, stats, out, o,
                           len, n);
                });
        };
        if (log_output) launch_all(std::true_type{});
        else launch_all(std::false_type{});
        after_launch("softmax_backward");
        p.done();
    });
}

}  // extern "C"
