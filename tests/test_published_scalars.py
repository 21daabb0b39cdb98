"""Sums and one-value scalar operations that publish their value as they are
computed: the value and the bits of the unpublished entry points, and item()
on a mean returning before the work enqueued after it has drained."""

import ctypes
import os

import numpy as np
import pytest

import vectorcore_amd as vc
from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu


def read(mirror):
    value = ctypes.c_float()
    C.check(C.lib().vc_hip_mirror_read(mirror, ctypes.byref(value)))
    C.check(C.lib().vc_hip_mirror_release(mirror))
    return np.float32(value.value)


@pytest.mark.parametrize("n", [0, 1, 5, 1025, 300_001])
@pytest.mark.parametrize("profiled", [False, True])
def test_published_sums_and_quotients(n, profiled):
    x = np.random.default_rng(n).standard_normal(n + 1).astype(np.float32)
    data = C.Buffer.of(x)
    plain, out, mirror = C.Buffer((1,)), C.Buffer((1,)), ctypes.c_void_p()
    C.profile(profiled)
    try:
        for start in (0, 4):  # on a 16-byte boundary and off it
            C.check(C.lib().vc_hip_reduce_sum(data.ptr + start, n, plain.ptr))
            C.check(C.lib().vc_hip_reduce_sum_published(data.ptr + start, n, out.ptr, ctypes.byref(mirror)))
            assert read(mirror) == out.numpy()[0] == plain.numpy()[0]
            for op in (C.ADD, C.SUB, C.MUL, C.DIV):
                for first in (0, 1):
                    C.check(C.lib().vc_hip_binary_scalar(out.ptr, 1, 3.7, first, plain.ptr, op))
                    C.check(C.lib().vc_hip_binary_scalar_published(out.ptr, 3.7, first, data.ptr, op, ctypes.byref(mirror)))
                    assert np.array_equal(read(mirror), plain.numpy()[0], equal_nan=True)
            data = C.Buffer.of(x)
    finally:
        C.profile(False)
    assert C.lib().vc_hip_reduce_sum_published(data.ptr, n, out.ptr, None) == 1
    assert C.lib().vc_hip_binary_scalar_published(data.ptr, 1.0, 0, out.ptr, 9, ctypes.byref(mirror)) == 1


@pytest.mark.skipif(os.environ.get("VECTORCORE_HIP_SYNC_EACH") == "1",
                    reason="every launch is waited for in this mode")
def test_a_means_value_does_not_wait_for_later_work():
    x = np.random.default_rng(0).standard_normal((1 << 20,)).astype(np.float32)
    t, a = vc.Tensor(x, device="hip"), vc.Tensor(np.ones((2048, 2048), np.float32), device="hip")
    vc.synchronize()
    mean = t.mean()
    for _ in range(100):
        a = (a @ a) * 0.0
    value = mean.item()
    assert not C.stream_idle()
    np.testing.assert_allclose(value, x.astype(np.float64).mean(), rtol=1e-5, atol=1e-9)
    vc.synchronize()
