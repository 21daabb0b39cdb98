"""Softmax and log-softmax as one node: both directions against float64, over
the kernels' edges (row lengths around what a wavefront holds, odd lengths,
columns, long rows), and what the composition did around them: special values,
in-place writes of the input between the passes, retained graphs."""

import numpy as np
import pytest

import vectorcore_amd as vc

pytestmark = pytest.mark.gpu


def exact(x, g, axis, log):
    x, g = x.astype(np.float64), g.astype(np.float64)
    shifted = x - x.max(axis, keepdims=True)
    total = np.exp(shifted).sum(axis, keepdims=True)
    p = np.exp(shifted) / total
    if log:
        return shifted - np.log(total), g - p * g.sum(axis, keepdims=True)
    return p, p * (g - (p * g).sum(axis, keepdims=True))


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("shape,axis", [((5, 1), 1), ((7, 3), 1), ((300, 10), 1), ((9, 255), 1), ((9, 256), 1),
                                        ((9, 257), 1), ((4, 511), -1), ((3, 1003), 1), ((2, 2048), 1), ((2, 2049), 1),
                                        ((3, 32000), 1), ((5, 70, 3), 1), ((64, 33, 20), 1), ((2, 513, 2048), 1),
                                        ((600, 5), 0), ((300, 4100), 0), ((2, 3, 4, 5), 2), ((17,), 0)])
def test_both_directions_against_float64(shape, axis, log):
    rng = np.random.default_rng(sum(shape) + axis)
    x = (2.0 * rng.standard_normal(shape)).astype(np.float32)
    g = rng.standard_normal(shape).astype(np.float32)
    t = vc.Tensor(x, requires_grad=True, device="hip")
    y = t.log_softmax(axis) if log else t.softmax(axis)
    y.backward(vc.Tensor(g, device="hip"))
    want_y, want_dx = exact(x, g, axis, log)
    # Per element a handful of roundings of values up to the shifted input's size, on which exp turns an
    # absolute error into a relative one: 24 covers the largest |x - m|.
    unit = 2.0 ** -24
    np.testing.assert_allclose(y.numpy(), want_y, rtol=64 * unit, atol=64 * unit * (np.abs(want_y).max() if log else 1.0))
    scale = np.abs(g).max() + np.abs(g.astype(np.float64)).sum(axis, keepdims=True) * (np.exp(want_y) if log else want_y)
    assert (np.abs(t.grad.numpy() - want_dx) <= 64 * unit * scale).all()


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("shape,axis", [((6, 7), 1), ((6, 2100), 1), ((7, 6), 0)])
def test_special_values_match_the_cpu_device(shape, axis, log):
    x = np.random.default_rng(3).standard_normal(shape).astype(np.float32)
    rows = x if axis == 1 else x.T
    rows[0, 2], rows[1, 3], rows[2, 0], rows[3, 4] = np.inf, -np.inf, np.nan, np.nan
    rows[4, :] = -np.inf
    rows[5, :] = np.finfo(np.float32).min
    got, want = [], []
    for out, device in ((got, "hip"), (want, "cpu")):
        t = vc.Tensor(np.ascontiguousarray(x), requires_grad=True, device=device)
        y = t.log_softmax(axis) if log else t.softmax(axis)
        y.backward(vc.Tensor(np.ones(shape, np.float32), device=device))
        out += [y.numpy(), t.grad.numpy()]
    for a, b in zip(got, want):
        np.testing.assert_allclose(a, b, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("log", [False, True])
def test_a_step_on_the_input_between_the_passes(log):
    """The composition saves nothing of its input: the rule's input is the one the forward saw."""
    x = np.random.default_rng(5).standard_normal((40, 33)).astype(np.float32)
    g = np.random.default_rng(6).standard_normal((40, 33)).astype(np.float32)
    grads = []
    for write in (False, True):
        t = vc.Tensor(x, requires_grad=True, device="hip")
        y = t.log_softmax(1) if log else t.softmax(1)
        if write:
            (t * 1.0).sum().backward()
            vc.sgd_step([t], 0.5)
            t.zero_grad()
        y.backward(vc.Tensor(g, device="hip"))
        grads.append(t.grad.numpy())
        if write:
            np.testing.assert_array_equal(t.numpy(), x - np.float32(0.5))
            y.backward(vc.Tensor(g, device="hip"))  # the graph is kept, as every graph is
            np.testing.assert_array_equal(t.grad.numpy(), grads[0] + grads[0])
    np.testing.assert_array_equal(grads[0], grads[1])


def test_softmax_refuses_its_modified_result_and_log_softmax_does_not():
    for log in (False, True):
        t = vc.Tensor(np.ones((4, 8), np.float32), requires_grad=True, device="hip")
        y = t.log_softmax(1) if log else t.softmax(1)
        y.retain_grad()
        g = vc.Tensor(np.ones((4, 8), np.float32), device="hip")
        y.backward(g)
        vc.sgd_step([y], 0.1)
        if log:
            y.backward(g)
        else:
            with pytest.raises(RuntimeError, match="modified in place"):
                y.backward(g)


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("shape", [(533, 16, 9), (534, 16, 9),  # on the two sides of the choice
                                   (70_000, 2, 2), (9000, 31, 3), (4000, 5, 70), (3, 4, 90_001), (20_000, 300, 2),
                                   (300_001, 1, 2), (1 << 23, 2, 2)])  # 2^23 workgroups of 512 could not be launched
def test_many_short_columns(shape, log):
    test_both_directions_against_float64(shape, 1, log)


@pytest.mark.parametrize("log", [False, True])
def test_special_values_in_short_columns_match_the_cpu_device(log):
    x = np.random.default_rng(4).standard_normal((1000, 5, 6)).astype(np.float32)
    x[0, 2, 1], x[1, 3, 2], x[2, 0, 3], x[3, 4, 4] = np.inf, -np.inf, np.nan, np.nan
    x[4, :, 5] = -np.inf
    x[5, :, 0] = np.finfo(np.float32).min
    got, want = [], []
    for out, device in ((got, "hip"), (want, "cpu")):
        t = vc.Tensor(x, requires_grad=True, device=device)
        y = t.log_softmax(1) if log else t.softmax(1)
        y.backward(vc.Tensor(np.ones(x.shape, np.float32), device=device))
        out += [y.numpy(), t.grad.numpy()]
    for a, b in zip(got, want):
        np.testing.assert_allclose(a, b, rtol=1e-5, atol=2e-6)
