"""The forward's elementwise ops of tensors that need a gradient: recorded, and
computed by the backward pass or by what reads them. Each case against the eager
ops (the same bits where no sum is involved) and the cpu device: results read
before, between and after backward passes, in-place writes of the inputs in
between, results nothing reads, expressions longer than a program, and a
forward that never runs backward."""

import time

import numpy as np
import pytest

import vectorcore_amd as vc
from vectorcore_amd import cabi as C

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(11)
X = RNG.standard_normal((130, 67)).astype(np.float32)
B = RNG.standard_normal((67,)).astype(np.float32)
DY = RNG.standard_normal((130, 67)).astype(np.float32)


def chain(x, b):
    return (x + b).relu().sigmoid() * (x * 0.1).exp() - (x * x + 1.0).log() / (-b).exp()


def pair(device="hip"):
    return (vc.Tensor(X, requires_grad=True, device=device), vc.Tensor(B, requires_grad=True, device=device))


@pytest.fixture(params=[True, False])
def fused(request):
    before = vc.hip_fuse_elementwise(request.param)
    yield request.param
    vc.hip_fuse_elementwise(before)


def outcome(order, device="hip"):
    x, b = pair(device)
    y = chain(x, b)
    out = [y.numpy()] if order == "read first" else []
    y.backward(vc.Tensor(DY, device=device))
    if order == "twice":
        y.backward(vc.Tensor(DY, device=device))
    return out + [y.numpy(), x.grad.numpy(), b.grad.numpy()]


@pytest.mark.parametrize("order", ["read first", "read after", "twice"])
def test_results_and_gradients(order, fused):
    got, cpu = outcome(order), outcome(order, "cpu")
    for a, c in zip(got, cpu):
        np.testing.assert_allclose(a, c, rtol=2e-5, atol=2e-5)
    before = vc.hip_fuse_elementwise(False)
    eager = outcome(order)
    vc.hip_fuse_elementwise(before)
    for a, e in zip(got[:-1], eager[:-1]):  # all but the column sum: the same bits
        np.testing.assert_array_equal(a, e)


def test_an_input_written_in_place_before_the_result_is_read(fused):
    x, b = pair()
    y, z = chain(x, b), x * 2.0
    (x * 1.0).sum().backward()
    vc.sgd_step([x], 0.5)  # bumps x's version
    np.testing.assert_array_equal(x.numpy(), X - np.float32(0.5))
    np.testing.assert_array_equal(z.numpy(), X * np.float32(2))  # what the ops saw
    np.testing.assert_allclose(y.numpy(), chain(*pair("cpu")).numpy(), rtol=2e-5, atol=2e-5)
    with pytest.raises(RuntimeError, match="modified in place"):
        y.backward(vc.Tensor(DY, device="hip"))


def test_intermediate_results_and_retained_gradients(fused):
    x, b = pair()
    h = (x + b).sigmoid()
    h.retain_grad()
    y = h * h
    y.backward(vc.Tensor(DY, device="hip"))
    s = 1 / (1 + np.exp(-(X.astype(np.float64) + B)))
    np.testing.assert_allclose(h.numpy(), s, rtol=1e-5)
    np.testing.assert_allclose(h.grad.numpy(), 2 * s * DY, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(x.grad.numpy(), 2 * s * DY * s * (1 - s), rtol=2e-5, atol=1e-6)


def test_a_chain_longer_than_a_program(fused):
    x, b = pair()
    cx, cb = pair("cpu")
    y, c = x, cx
    for i in range(40):
        y = (y * 0.9 + b).sigmoid() if i % 5 == 4 else y * 0.9 + b
        c = (c * 0.9 + cb).sigmoid() if i % 5 == 4 else c * 0.9 + cb
    y.backward(vc.Tensor(DY, device="hip"))
    c.backward(vc.Tensor(DY))
    np.testing.assert_allclose(y.numpy(), c.numpy(), rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(x.grad.numpy(), cx.grad.numpy(), rtol=1e-3, atol=1e-7)


@pytest.mark.parametrize("length", [15, 16, 17, 33])
def test_chains_about_the_longest_recorded_one(length):
    """The next operation's operand is computed then; every result and gradient has the eager ops' bits."""
    outcomes = []
    for fuse in (True, False):
        before = vc.hip_fuse_elementwise(fuse)
        x = vc.Tensor(X, requires_grad=True, device="hip")
        y, results = x, []
        for k in range(length):
            y = (y * 1.25, y.sigmoid(), y - 0.5, y.relu(), y * y)[k % 5] if k % 3 else y * y + y * 0.5
            results.append(y)
        y.backward(vc.Tensor(DY, device="hip"))
        outcomes.append([r.numpy() for r in results[::4]] + [y.numpy(), x.grad.numpy()])
        vc.hip_fuse_elementwise(before)
    for a, b in zip(*outcomes):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("shape", [(1,), (3,), (2, 1), (1, 5), (2, 3, 4), (1025,)])
def test_shapes_and_no_backward(shape, fused):
    x = RNG.standard_normal(shape).astype(np.float32)
    t = vc.Tensor(x, requires_grad=True, device="hip")
    np.testing.assert_array_equal((-(t.relu() + 1.0)).numpy(), -(np.maximum(x, 0) + np.float32(1)))
    np.testing.assert_array_equal((t * t).T.numpy() if len(shape) > 1 else (t * t).numpy(),
                                  np.swapaxes(x * x, -1, -2) if len(shape) > 1 else x * x)
    assert abs((t * 3.0).sum().item() - float((x * np.float32(3)).astype(np.float64).sum())) < 1e-3
    np.testing.assert_array_equal((t * t).max(0).numpy(), (x * x).max(0))
    with np.errstate(all="ignore"):
        np.testing.assert_allclose(t.log().numpy(), np.log(x), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("rows,cols,recorded", [(16_384, 3, True), (16_385, 3, False), (20_000, 127, False),
                                                (20_000, 128, True)])
def test_many_short_rows_are_summed_by_the_reduction(rows, cols, recorded):
    x = RNG.standard_normal((rows, cols)).astype(np.float32)
    w = RNG.standard_normal((rows, 1)).astype(np.float32)
    t, tw = (vc.Tensor(v, requires_grad=True, device="hip") for v in (x, w))
    fuse = vc.hip_fuse_elementwise(True)
    C.profile(True)
    C.profile_reset()
    try:
        s = (t * tw).sum(1)  # the row sum of a forward expression, and of a gradient (w's)
        s.backward(vc.Tensor(np.ones(rows, np.float32), device="hip"))
        got = s.numpy(), tw.grad.numpy(), t.grad.numpy()
        assert ("fused_map_rows" in C.profile_read()) == recorded
    finally:
        C.profile(False)
        vc.hip_fuse_elementwise(fuse)
    np.testing.assert_allclose(got[0], (x * w).astype(np.float64).sum(1), rtol=2e-7, atol=1e-9)
    np.testing.assert_allclose(got[1], x.astype(np.float64).sum(1, keepdims=True), rtol=2e-7, atol=1e-9)
    np.testing.assert_array_equal(got[2], np.broadcast_to(w, x.shape))


def test_recording_a_chain_costs_no_more_than_launching_it():
    """Small operands: the host's work is the pass's time. Recorded, about half of it (measured 244 against 516 us)."""
    x = vc.Tensor(X[:16, :64], requires_grad=True, device="hip")
    g = vc.Tensor(DY[:16, :64], device="hip")

    def seconds(fuse):
        before = vc.hip_fuse_elementwise(fuse)
        best = float("inf")
        for _ in range(20):
            vc.synchronize()
            start = time.perf_counter()
            y = x
            for k in range(32):
                y = y * 0.9 if k % 4 == 0 else y.sigmoid() if k % 2 else y + x
            y.backward(g)
            vc.synchronize()
            best = min(best, time.perf_counter() - start)
            x.zero_grad()
        vc.hip_fuse_elementwise(before)
        return best

    assert seconds(True) < seconds(False)
