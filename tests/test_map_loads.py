"""How matrix programs (vc_hip_map_broadcast) load their inputs: one value per
element, column, row and group in one program, over matrices whose rows are
shorter than a vector, whole vectors and not, one row, one column, groups of one
row, several workgroups, and inputs on odd 4-byte boundaries; without sums, with
row sums and with column sums. And the sigmoid's two sides, as programs and the
eager kernel compute them."""

import ctypes

import numpy as np
import pytest

import vectorcore_amd as vc
from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 9, 1), (9, 1, 3), (6, 2, 1), (6, 3, 2), (6, 4, 6), (10, 8, 5), (12, 63, 3), (12, 64, 4), (40, 260, 8),
          (2100, 12, 7), (9, 1003, 9), (3, 4100, 1), (4, 5001, 2), (515, 1028, 5)]


def offset_buffer(values, offset):
    """A device buffer that holds the values from 4 * offset bytes on."""
    return C.Buffer.of(np.concatenate([np.full(offset, np.nan, np.float32), values.ravel()]))


@pytest.mark.parametrize("rows,cols,length", SHAPES)
@pytest.mark.parametrize("sums", ["none", "rows", "columns"])
@pytest.mark.parametrize("offset", [0, 1])
def test_every_kind_of_input(rows, cols, length, sums, offset):
    rng = np.random.default_rng(rows * cols + length)
    full, column, row, group = (rng.integers(-9, 10, size=s).astype(np.float32)
                                for s in ((rows, cols), (1, cols), (rows, 1), (rows // length, 1, cols)))
    want = full + (column * row - np.broadcast_to(group, (rows // length, length, cols)).reshape(rows, cols))
    bufs = [offset_buffer(v, offset) for v in (full, column, row, group)]
    out, total = C.Buffer((rows * cols,)), C.Buffer((max(rows, cols),))
    code = [(C.MAP_MUL, 1, 2, 4), (C.MAP_SUB, 4, 3, 4), (C.MAP_ADD, 0, 4, 5)]
    at = [b.ptr.value + 4 * offset if isinstance(b.ptr, ctypes.c_void_p) else b.ptr + 4 * offset for b in bufs]
    p = C.map_program(at, [], code, [(out.ptr, 5)], [(total.ptr, 5)] if sums == "columns" else [], rows, cols)
    m = C.MapMatrix()
    m.axis_length = length
    for j, kind in enumerate((C.MAP_FULL, C.MAP_PER_COLUMN, C.MAP_PER_ROW, C.MAP_PER_GROUP)):
        m.input_kinds[j] = kind
    if sums == "rows":
        m.row_sums[0], m.row_sum_slots[0], m.n_row_sums = total.ptr, 5, 1
    C.check(C.lib().vc_hip_map_broadcast(ctypes.byref(p), ctypes.byref(m)))
    np.testing.assert_array_equal(out.numpy().reshape(rows, cols), want)  # small whole numbers: exact in any order
    if sums == "rows":
        np.testing.assert_array_equal(total.numpy().ravel()[:rows], want.sum(1))
    if sums == "columns":
        np.testing.assert_array_equal(total.numpy().ravel()[:cols], want.sum(0))


def test_sigmoid_on_both_sides():
    x = np.array([0.0, -0.0, 1e-30, -1e-30, 1.0, -1.0, 17.5, -17.5, 88.0, -88.0, 104.0, -104.0, 3e38, -3e38, np.inf, -np.inf,
                  np.nan], np.float32)
    t = vc.Tensor(np.repeat(x, 16), device="hip", requires_grad=True)
    y = t.sigmoid()
    y.backward(vc.Tensor(np.ones(x.size * 16, np.float32), device="hip"))
    eager = vc.Tensor(np.repeat(x, 16), device="hip").sigmoid().numpy()
    np.testing.assert_array_equal(y.numpy(), eager)  # the same function in both kernels
    with np.errstate(over="ignore"):
        e = np.exp(-np.abs(np.repeat(x, 16).astype(np.float64)))
        want = np.where(np.repeat(x, 16) >= 0, 1.0, e) / (1.0 + e)
    # expf, the sum and the quotient: 1 + 0.5 + 0.5 ulp of 2^-23 each; below 2^-126 in whole steps of 2^-149.
    np.testing.assert_allclose(eager, want, rtol=4 * 2.0 ** -23, atol=2.0 ** -148)


def test_divided_by_a_host_scalar_along_an_axis():
    """The gradient of a mean: the quotient by a host-known count joins a program as a constant."""
    x = np.random.default_rng(3).standard_normal((33, 70)).astype(np.float32)
    grads = []
    for device in ("hip", "cpu"):
        t = vc.Tensor(x, device=device, requires_grad=True)
        y = (t / vc.Tensor(np.array([7.0], np.float32), device=device)) * t.mean(1, True)
        y.backward(vc.Tensor(np.cos(x), device=device))
        grads.append(t.grad.numpy())
    np.testing.assert_allclose(grads[0], grads[1], rtol=2e-5, atol=2e-6)


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 7, 1023, 1025, 4096 * 256 * 4 + 3])
def test_flat_programs_end_with_the_count(count):
    """The last vector of a count that is no multiple of 4 is moved back; nothing past the count is written."""
    x = np.random.default_rng(count).standard_normal(count).astype(np.float32)
    a, out = C.Buffer.of(x), C.Buffer.of(np.full(count + 4, 5.0, np.float32))
    p = C.map_program([a.ptr], [3.0], [(C.MAP_MUL, 0, 1, 2), (C.MAP_ADD, 2, 0, 3)], [(out.ptr, 3)], [], 1, count)
    C.check(C.lib().vc_hip_map(ctypes.byref(p)))
    np.testing.assert_array_equal(out.numpy(), np.concatenate([x * np.float32(3.0) + x, np.full(4, 5.0, np.float32)]))
