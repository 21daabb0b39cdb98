"""Products whose operands' rows are not whole 16-byte groups, and products of
few rows or tiles, whose K is split over waves and workgroups.

Each operand lies between NaNs, one float past a 16-byte boundary: a value read
from outside a matrix, or kept past K, would make an output NaN. Outputs are
compared with the float64 product; the bound is that of any order of k fp32
additions and multiplications, k 2^-23 times the product of the magnitudes."""

import numpy as np
import pytest

from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu

TRANSPOSES = ((0, 0), (1, 0), (0, 1), (1, 1))


def between_nans(x):
    """x on the device between NaNs, starting 4 bytes past a 16-byte boundary: (buffer, pointer)."""
    flat = np.full(x.size + 64, np.nan, np.float32)
    flat[33:33 + x.size] = x.ravel()
    buffer = C.Buffer.of(flat)
    return buffer, buffer.ptr + 33 * 4


def operands(m, k, n, ta, tb, batch, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1, 1, size=(batch,) + ((k, m) if ta else (m, k))).astype(np.float32)
    b = rng.uniform(-1, 1, size=(batch,) + ((n, k) if tb else (k, n))).astype(np.float32)
    wide_a = (a.transpose(0, 2, 1) if ta else a).astype(np.float64)
    wide_b = (b.transpose(0, 2, 1) if tb else b).astype(np.float64)
    return a, b, wide_a @ wide_b, np.abs(wide_a) @ np.abs(wide_b)


def check(got, want, magnitude, k, what):
    excess = np.abs(got - want) - (k * 2.0 ** -23 * magnitude + 1e-30)
    assert not np.isnan(got).any() and excess.max() <= 0, (what, excess.max())


# One to three values past a whole group along each of m, n and k; K of less
# than a group, of one chunk of 32, one past it, of fewer and more chunks than
# waves; tiles of one row and one column; K split over workgroups (few tiles).
@pytest.mark.parametrize("m,k,n", [(33, 3, 65), (129, 33, 35), (70, 35, 130), (31, 126, 63), (65, 131, 97),
                                   (1, 1001, 1003), (1003, 1001, 1), (2, 4099, 515), (33, 8193, 34), (515, 999, 131),
                                   (1, 4096, 1000), (16, 2048, 1024)])
def test_small_products_of_any_row_length(m, k, n):
    for ta, tb in TRANSPOSES:
        a, b, want, magnitude = operands(m, k, n, ta, tb, 1, m + k + n)
        (_a, pa), (_b, pb) = between_nans(a), between_nans(b)
        c = C.Buffer((1, m, n))
        z = C.sizes([0])
        C.check(C.lib().vc_hip_matmul(pa, pb, c.ptr, m, k, n, z, z, 1, ta, tb))
        first = c.numpy()
        check(first, want, magnitude, k, (ta, tb))
        C.check(C.lib().vc_hip_matmul(pa, pb, c.ptr, m, k, n, z, z, 1, ta, tb))
        np.testing.assert_array_equal(c.numpy(), first)  # the split ranges are added in one order


# Partial tiles and K tails of one to three values on the 256-row tiles, with
# K of less than a slice, one slice and a value, and several.
@pytest.mark.parametrize("kernel", ["mfma128", "mfma256", "mfma256x128"])
@pytest.mark.parametrize("m,k,n", [(257, 31, 129), (259, 33, 513), (511, 98, 255), (130, 163, 259)])
def test_large_tiles_of_any_row_length(kernel, m, k, n):
    for ta, tb in TRANSPOSES:
        a, b, want, magnitude = operands(m, k, n, ta, tb, 2, m + k + n)
        (_a, pa), (_b, pb) = between_nans(a), between_nans(b)
        c = C.Buffer((2, m, n))
        with C.gemm_kernel(kernel):
            C.check(C.lib().vc_hip_matmul(pa, pb, c.ptr, m, k, n, C.sizes([0, m * k]), C.sizes([0, k * n]), 2, ta, tb))
        check(c.numpy(), want, magnitude, k, (ta, tb))


# The choice between the 256-row and the 32 x 32 tiles, either side of it.
@pytest.mark.parametrize("m,k,n", [(4095, 65, 2047), (2047, 65, 2047), (1501, 701, 903)])
def test_odd_products_on_both_sides_of_the_tile_choice(m, k, n):
    for ta, tb in TRANSPOSES:
        a, b, want, magnitude = operands(m, k, n, ta, tb, 1, m + k + n)
        (_a, pa), (_b, pb) = between_nans(a), between_nans(b)
        c = C.Buffer((1, m, n))
        z = C.sizes([0])
        C.check(C.lib().vc_hip_matmul(pa, pb, c.ptr, m, k, n, z, z, 1, ta, tb))
        check(c.numpy(), want, magnitude, k, (ta, tb))


# A batch reduction: the chunks of each product follow those of the one before, ranges may begin inside one.
@pytest.mark.parametrize("m,k,n,count", [(65, 197, 131, 48), (33, 31, 33, 7), (130, 64, 60, 5)])
def test_batch_reduction_of_any_row_length(m, k, n, count):
    for ta, tb in TRANSPOSES:
        a, b, want, magnitude = operands(m, k, n, ta, tb, count, m + k + n)
        (_a, pa), (_b, pb) = between_nans(a), between_nans(b)
        c = C.Buffer((m, n))
        C.check(C.lib().vc_hip_matmul_reduce(pa, pb, c.ptr, m, k, n, count, m * k, k * n, ta, tb))
        check(c.numpy(), want.sum(0), magnitude.sum(0), k * count, (ta, tb))


# The epilogues after a split K: bias and ReLU, the mask as floats and as bits, the column sums.
@pytest.mark.parametrize("m,k,n", [(33, 1001, 35), (70, 2047, 130)])
def test_split_products_keep_their_epilogues(m, k, n):
    rng = np.random.default_rng(m)
    a, b, want, magnitude = operands(m, k, n, 0, 0, 1, m + k + n)
    (_a, pa), (_b, pb) = between_nans(a), between_nans(b)
    bias, mask = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    plain, c = C.Buffer((m, n)), C.Buffer((m, n))
    z, zero = C.sizes([0]), np.float32(0)
    C.check(C.lib().vc_hip_matmul(pa, pb, plain.ptr, m, k, n, z, z, 1, 0, 0))
    product = plain.numpy()
    check(product[None], want, magnitude, k, "plain")
    C.check(C.lib().vc_hip_matmul_bias_relu(pa, pb, c.ptr, m, k, n, C.Buffer.of(bias).ptr, 1))
    np.testing.assert_array_equal(c.numpy(), np.where(product + bias > 0, product + bias, zero))
    masked = product * (mask > 0).astype(np.float32)
    sums = C.Buffer((n,))
    device_mask = C.Buffer.of(mask)
    C.check(C.lib().vc_hip_matmul_relu_mask_colsum(pa, pb, c.ptr, m, k, n, 0, 0, device_mask.ptr, sums.ptr))
    np.testing.assert_array_equal(c.numpy(), masked)
    np.testing.assert_allclose(sums.numpy(), masked.astype(np.float64).sum(0), rtol=2e-7, atol=1e-6)
    words = np.zeros(((m + 31) // 32, n), np.uint32)
    for r in range(m):
        words[r // 32] |= (mask[r] > 0).astype(np.uint32) << np.uint32(r % 32)
    C.check(C.lib().vc_hip_matmul_relu_bits(pa, pb, c.ptr, m, k, n, 0, 0, C.Buffer.of(words, dtype=np.uint32).ptr))
    np.testing.assert_array_equal(c.numpy(), masked)


@pytest.mark.parametrize("count,m,k,n", [(32, 768, 768, 768), (64, 512, 512, 512), (16, 1024, 512, 1024)])
def test_reductions_of_many_outputs_take_the_large_tiles(count, m, k, n):
    """A sum over many products is as much work as one product of count k: the 128 x 128 tiles, split over the
    products, add in another order than the 32 x 32 tiles, so their bits tell which kernel ran."""
    rng = np.random.default_rng(count)
    a = C.Buffer.of(rng.standard_normal((count, k, m)).astype(np.float32))
    b = C.Buffer.of(rng.standard_normal((count, k, n)).astype(np.float32))
    c = C.Buffer((m, n))
    results = []
    for kernel in ("mfma", "mfma128"):
        with C.gemm_kernel(kernel):
            C.check(C.lib().vc_hip_matmul_reduce(a.ptr, b.ptr, c.ptr, m, k, n, count, k * m, k * n, 1, 0))
        results.append(c.numpy())
    np.testing.assert_array_equal(*results)


@pytest.mark.parametrize("batch,m,k,n,tb", [(2, 1544, 36, 1160, 1), (8, 12960, 12, 48, 0), (1, 512, 48, 4736, 0)])
def test_short_k_of_many_outputs_takes_the_large_tiles(batch, m, k, n, tb):
    """About one round of 128 x 128 tiles and a K of one or two chunks: the small tiles' fixed cost decides."""
    a, b, want, magnitude = operands(m, k, n, 0, tb, batch, k)
    a, b, c = C.Buffer.of(a), C.Buffer.of(b), C.Buffer((batch, m, n))
    za, zb = C.sizes([m * k * z for z in range(batch)]), C.sizes([k * n * z for z in range(batch)])
    results = []
    for kernel in ("mfma", "mfma128"):
        with C.gemm_kernel(kernel):
            C.check(C.lib().vc_hip_matmul(a.ptr, b.ptr, c.ptr, m, k, n, za, zb, batch, 0, tb))
        results.append(c.numpy())
    np.testing.assert_array_equal(*results)
    check(results[0], want, magnitude, k, (batch, m, k, n))
