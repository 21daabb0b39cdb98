"""Max and argmax along an axis, singly and from one pass, over the column
kernel's edges: columns around its 16 and 64, axes around its row lanes and
loads in flight, few and many workgroups, axes long enough to be split, and the
scan's special values (the first maximum wins, NaN never does but first)."""

import numpy as np
import pytest

from oracle import kernels as K
from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu


def reduce(x, shape, op):
    out = C.Buffer((shape[0], shape[2]))
    C.check(C.lib().vc_hip_reduce_axis(x, out.ptr, *shape, op))
    return out.numpy()


@pytest.mark.parametrize("shape", [(3, 15, 5), (3, 16, 5), (2, 17, 63), (2, 128, 64), (2, 129, 65), (200, 40, 67),
                                   (64, 197, 96), (1, 1024, 17), (1, 1025, 17), (1, 5000, 3), (130, 1100, 30), (5, 1, 9),
                                   (70, 33, 1), (3, 1003, 1), (400, 20, 130)])
def test_both_reductions_match_the_scan(shape):
    rng = np.random.default_rng(sum(shape))
    x = rng.integers(-4, 5, size=shape).astype(np.float32)  # with ties
    flat = x.reshape(-1)
    flat[rng.random(flat.size) < 0.05] = np.nan
    flat[rng.random(flat.size) < 0.05] = -np.inf
    flat[rng.random(flat.size) < 0.02] = np.inf
    x[0, :, 0] = -np.inf
    x[-1, 0, -1] = np.nan
    buffer = C.Buffer.of(np.concatenate([np.zeros(1, np.float32), flat]))
    for start in (0, 4):  # on a 16-byte boundary and off it
        data = C.Buffer.of(flat) if start == 0 else buffer
        want_max, want_arg = K.reduce_axis(x, 1, K.MAX), K.reduce_axis(x, 1, K.ARGMAX)
        best, where = C.Buffer((shape[0], shape[2])), C.Buffer((shape[0], shape[2]))
        C.check(C.lib().vc_hip_reduce_axis_max_argmax(data.ptr + start, best.ptr, where.ptr, *shape))
        for got, want in ((best.numpy(), want_max), (where.numpy(), want_arg),
                          (reduce(data.ptr + start, shape, C.MAX), want_max),
                          (reduce(data.ptr + start, shape, C.ARGMAX), want_arg)):
            np.testing.assert_array_equal(got.reshape(-1), np.asarray(want).reshape(-1))


def test_an_empty_axis_and_null_outputs_are_refused():
    x = C.Buffer((4,))
    with pytest.raises(ValueError):
        C.check(C.lib().vc_hip_reduce_axis_max_argmax(x.ptr, x.ptr, x.ptr, 2, 0, 2))
    with pytest.raises(ValueError):
        C.check(C.lib().vc_hip_reduce_axis_max_argmax(x.ptr, x.ptr, None, 1, 2, 2))


@pytest.mark.parametrize("shape", [(5000, 16, 2), (30_000, 17, 3), (100_000, 16, 16), (16, 16, 8000), (4096, 24, 100),
                                   (10_000, 64, 2), (20_000, 100, 2), (1024, 63, 63), (4096, 63, 63), (2000, 197, 8)])
def test_short_and_narrow_columns_match_the_scan(shape):
    """Shapes about where a workgroup of row lanes, a thread per column and a split axis take over from each other."""
    test_both_reductions_match_the_scan(shape)
