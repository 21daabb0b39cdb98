"""Backward passes whose operands broadcast, through matrix programs
(vc_hip_map_broadcast): each gradient against the cpu device, which evaluates
the rules one op at a time, over the ways an operand broadcasts (per column, per
row, per group, one value, ways that no matrix view serves), rows shorter than
a vector, odd lengths and conflicting views; then the entry point's checks."""

import ctypes

import numpy as np
import pytest

import vectorcore_amd as vc
from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu

SHAPES = [((6, 5), (5,)), ((6, 5), (6, 1)), ((6, 5), (1, 5)), ((6, 5), (1, 1)), ((7, 3), (7, 1)), ((9, 2), (2,)),
          ((130, 1003), (1003,)), ((130, 1003), (130, 1)), ((3000, 33), (3000, 1)), ((5, 7, 9), (5, 1, 9)),
          ((5, 7, 9), (7, 1)), ((5, 7, 9), (5, 1, 1)), ((5, 7, 9), (1, 7, 1)), ((2, 3, 4, 5), (2, 1, 4, 1)),
          ((4, 1, 6), (4, 1, 1)), ((1, 8), (1, 1)), ((2100, 4), (2100, 1)), ((40, 4100), (40, 1))]


def both(build, *arrays):
    """[outputs on hip], [outputs on cpu] of build(device, *arrays)."""
    return [build(d, *arrays) for d in ("hip", "cpu")]


def grads(device, f, arrays, dy):
    ts = [vc.Tensor(a, requires_grad=True, device=device) for a in arrays]
    y = f(*ts)
    y.backward(vc.Tensor(dy(y.shape), device=device))
    return [t.grad.numpy() for t in ts] + [y.numpy()]


def compare(f, arrays):
    rng = np.random.default_rng(7)
    made = {}

    def dy(shape):
        return made.setdefault(tuple(shape), rng.standard_normal(tuple(shape)).astype(np.float32))

    want, got = grads("cpu", f, arrays, dy), grads("hip", f, arrays, dy)
    for a, b in zip(got, want):
        assert a.shape == b.shape
        # The same fp32 operations per element; sums in double on both, exp and log to 1e-6 relative.
        np.testing.assert_allclose(a, b, rtol=2e-5, atol=2e-6 * max(1.0, float(np.abs(b).max())))


@pytest.mark.parametrize("big,small", SHAPES)
def test_broadcast_gradients_match_the_cpu_device(big, small):
    rng = np.random.default_rng(len(big) + sum(big))
    a = rng.standard_normal(big).astype(np.float32)
    b = (np.abs(rng.standard_normal(small)) + 0.5).astype(np.float32)
    compare(lambda x, y: x * y + y, [a, b])
    compare(lambda x, y: (x - y) / y, [a, b])
    compare(lambda x, y: y / (x * x + 1.0) - x * y, [a, b])


@pytest.mark.parametrize("shape", [(33, 70), (1, 5), (5, 1), (64, 1024), (2050, 1030), (7, 3)])
def test_rows_brought_to_mean_0_and_variance_1(shape):
    rng = np.random.default_rng(sum(shape))

    def f(x, gain, offset):
        c = x - x.mean(1, True)
        return c / (((c * c).mean(1, True) + 1e-3).log() * 0.5).exp() * gain + offset

    compare(f, [rng.standard_normal(shape).astype(np.float32), rng.standard_normal(shape[1]).astype(np.float32),
                rng.standard_normal(shape[1]).astype(np.float32)])


@pytest.mark.parametrize("shape", [(6, 7, 8), (1, 9, 5), (33, 2, 3), (5, 300, 1), (4, 1, 9), (3, 65, 130)])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("keepdim", [False, True])
def test_maximum_and_mean_along_an_axis(shape, axis, keepdim):
    x = np.random.default_rng(axis + sum(shape)).integers(-3, 4, size=shape).astype(np.float32)  # with ties
    compare(lambda t: t.max(axis, keepdim) + t.mean(axis, keepdim) * 2.0, [x])
    compare(lambda t: t.max(axis, True) * t, [x])


def test_views_that_disagree_are_computed_apart():
    rng = np.random.default_rng(1)
    x = rng.standard_normal((6, 4, 10)).astype(np.float32)
    a, b, c = (rng.standard_normal(s).astype(np.float32) for s in ((6, 1, 10), (1, 4, 1), (6, 4, 1)))
    compare(lambda x, a, b, c: ((x * a) * b) * c + x.max(1, True) * a, [x, a, b, c])


def matrix_program(**change):
    x, out = C.Buffer.of(np.arange(12, dtype=np.float32)), C.Buffer((12,))
    vector, rows = C.Buffer.of(np.arange(4, dtype=np.float32)), C.Buffer((3,))
    p = C.map_program([x.ptr, vector.ptr], [], [(C.MAP_MUL, 0, 1, 2)], [(out.ptr, 2)], [], change.get("rows", 3),
                      change.get("cols", 4))
    m = C.MapMatrix()
    m.input_kinds[1] = change.get("kind", C.MAP_PER_COLUMN)
    m.axis_length = change.get("axis", 1)
    if change.get("row_sums"):
        m.row_sums[0], m.row_sum_slots[0], m.n_row_sums = rows.ptr, change.get("slot", 2), change["row_sums"]
    return p, m, out, rows, (x, vector)


def test_entry_point_computes_and_refuses():
    p, m, out, rows, keep = matrix_program(row_sums=1)
    C.check(C.lib().vc_hip_map_broadcast(ctypes.byref(p), ctypes.byref(m)))
    want = np.arange(12, dtype=np.float32).reshape(3, 4) * np.arange(4, dtype=np.float32)
    np.testing.assert_array_equal(out.numpy().reshape(3, 4), want)
    np.testing.assert_array_equal(rows.numpy(), want.sum(1))
    for change in ({"kind": 4}, {"axis": 2}, {"axis": 0}, {"rows": 0}, {"cols": 0}, {"rows": 1 << 30}, {"row_sums": 3},
                   {"row_sums": 1, "slot": 9}):
        p, m, out, rows, keep = matrix_program(**change)
        with pytest.raises(ValueError):
            C.check(C.lib().vc_hip_map_broadcast(ctypes.byref(p), ctypes.byref(m)))
    p, m, out, rows, keep = matrix_program()
    p.code[0] = C.map_word(C.MAP_AT_COLUMN, 0, 1, 2)
    with pytest.raises(ValueError):
        C.check(C.lib().vc_hip_map(ctypes.byref(p)))  # positions need a matrix
