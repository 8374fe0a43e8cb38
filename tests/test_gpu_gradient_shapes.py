"""The weight- and bias-gradient reductions at the shapes where their split of
the work can go wrong: one run of rows shorter than a workgroup's step, a last
run cut short, several 64-pixel bands, one image and several, more tasks than
workgroups.

Bounds: the CPU oracle rounds to BF16 where the kernels do, so the two differ
by the order of FP32 sums and by single BF16 roundings of activations at a
rounding boundary (2^-9 relative each, averaged over the pixels): 2e-2 per
block of the gradient, as for the shape the trainer is checked at elsewhere.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch  # noqa: F401

from conftest import REPO

sys.path.insert(0, str(REPO / "oracle"))
import cnn_oracle as co  # noqa: E402
from tealeaf_cuda_amd import warmstart as wsm  # noqa: E402

pytestmark = pytest.mark.gpu


def _blocks():
    out = [("w1", co.OFF_W1, co.OFF_B1), ("b1", co.OFF_B1, co.OFF_HID)]
    for l in range(4):
        o = co.OFF_HID + l * co.HID
        w = o + co.TAPS * co.CH * co.CH
        out += [(f"w{l + 2}", o, w), (f"b{l + 2}", w, o + co.HID)]
    return out + [("w6", co.OFF_W6, co.OFF_B6), ("b6", co.OFF_B6, co.NPARAM)]


@pytest.mark.parametrize("shape", [(1, 4, 64), (3, 12, 64), (2, 20, 192), (1, 36, 128), (40, 8, 64)])
def test_gradient_at_odd_shapes(shape):
    print(f"[gpu gradient] batch, height, width {shape}", flush=True)
    b, h, w = shape
    rng = np.random.default_rng(11)
    params = co.init_params(3).astype(np.float64)
    params[co.OFF_W6:] = 0.1 * rng.standard_normal(co.NPARAM - co.OFF_W6)
    params = params.astype(np.float32)
    samples = rng.standard_normal((b, 6, h, w)).astype(np.float32)
    samples[:, 4:] = np.abs(samples[:, 4:])
    t = wsm.Trainer(b, h, w, margin=1, loss="energy")
    try:
        t.set_params(params)
        device = torch.from_numpy(samples).cuda()
        loss, grad = t.gradient(device)
        again, grad2 = t.gradient(device)
        assert loss == again and np.array_equal(grad, grad2)      # a fixed order of sums
        want_loss, want = co.loss_and_grad(params, samples, margin=1, mode="bf16", loss="energy")
        assert loss == pytest.approx(want_loss, rel=1e-3)
        for name, lo, hi in _blocks():
            scale = np.linalg.norm(want[lo:hi])
            assert np.linalg.norm(grad[lo:hi] - want[lo:hi]) < 2e-2 * scale, name
    finally:
        t.close()


SHAPES = [(1, 4, 64, 0), (1, 68, 128, 32), (2, 80, 192, 32), (4, 32, 64, 0), (1, 64, 64, 0), (1, 128, 128, 0),
          (8, 128, 128, 0), (64, 8, 64, 0)]


@pytest.mark.parametrize("loss", ["mse", "energy"])
@pytest.mark.parametrize("shape", SHAPES)
def test_gradient_of_whole_numbers(shape, loss):
    """Every entry of the gradient, exactly.  Weights of 0 and +-1 (one per
    output channel of the hidden layers, one per input channel of the last)
    and inputs, biases, errors and couplings of small whole numbers keep every
    activation below 9 and every gradient below 10 in units of 2 / |M|, a
    power of two at these shapes: all of them are BF16 values, and every sum
    is a whole number below 2^24 whatever its order."""
    b, h, w, margin = shape
    print(f"[gpu gradient] whole numbers, {shape}, {loss}", flush=True)
    rng = np.random.default_rng(5)
    signs = [-1.0, 1.0, 1.0, 1.0]
    w1 = np.zeros((co.K1, co.CH))
    w1[rng.integers(0, co.K1, co.CH), np.arange(co.CH)] = rng.choice([-1.0, 1.0], co.CH)
    hidden = []
    for _ in range(4):
        wl = np.zeros((co.TAPS, co.CH, co.CH))
        wl[rng.integers(0, co.TAPS, co.CH), rng.permutation(co.CH), np.arange(co.CH)] = rng.choice(signs, co.CH)
        hidden.append((wl, np.ones(co.CH)))
    w6 = np.zeros((co.TAPS, co.CH))
    w6[rng.integers(0, co.TAPS, co.CH), np.arange(co.CH)] = rng.choice([-1.0, 1.0], co.CH)
    params = co.pack(w1, np.ones(co.CH), hidden, w6, 1.0).astype(np.float32)
    samples = np.zeros((b, 6, h, w), dtype=np.float32)
    samples[:, :3] = rng.integers(-2, 3, (b, 3, h, w))
    samples[:, 4:] = rng.integers(0, 2, (b, 2, h, w))
    t = wsm.Trainer(b, h, w, margin=margin, loss=loss)
    try:
        t.set_params(params)
        out = t.forward(torch.from_numpy(samples).cuda()).reshape(b, h, w)
        samples[:, 3] = out - rng.integers(-1, 2, (b, h, w))      # errors of -1, 0, 1
        got_loss, grad = t.gradient(torch.from_numpy(samples).cuda())
    finally:
        t.close()
    want_loss, want = co.loss_and_grad(params, samples, margin=margin, mode="bf16", loss=loss)
    assert got_loss == want_loss
    for name, lo, hi in _blocks():
        assert np.any(want[lo:hi] != 0.0) and np.array_equal(grad[lo:hi], want[lo:hi].astype(np.float32)), name


@pytest.mark.parametrize("loss", ["mse", "energy"])
@pytest.mark.parametrize("shape", [(1, 4, 64, 1), (2, 20, 192, 1), (7, 52, 64, 3), (8, 128, 128, 6)])
def test_output_bias_is_summed_in_its_order(shape, loss):
    """The gradient of the output bias is the FP32 sum of the output's gradient
    over 256 runs of consecutive pixels, each from its first pixel to its last,
    then over the runs in turn: bit for bit (under the energy loss the values
    cancel in this sum, so another order is another error)."""
    b, h, w, m = shape
    print(f"[gpu gradient] output bias, {shape}, {loss}", flush=True)
    rng = np.random.default_rng(17)
    f = np.float32
    params = co.init_params(3).astype(np.float64)
    params[co.OFF_W6:] = 0.1 * rng.standard_normal(co.NPARAM - co.OFF_W6)
    samples = rng.standard_normal((b, 6, h, w)).astype(f)
    samples[:, 4:] = 10.0 * np.abs(samples[:, 4:])
    t = wsm.Trainer(b, h, w, margin=m, loss=loss)
    try:
        t.set_params(params.astype(f))
        device = torch.from_numpy(samples).cuda()
        out = t.forward(device).reshape(b, h, w)
        _, grad = t.gradient(device)
    finally:
        t.close()
    e = (out - samples[:, 3]).astype(f)
    ae = e.copy()
    if loss == "energy":
        y, x = np.arange(h)[:, None], np.arange(w)[None, :]
        kx, ky = samples[:, 4], samples[:, 5]
        for face, shift, axis, there in ((kx, 1, 2, x - 1 >= m), (np.roll(kx, -1, 2), -1, 2, x + 1 < w - m),
                                         (ky, 1, 1, y - 1 >= m), (np.roll(ky, -1, 1), -1, 1, y + 1 < h - m)):
            ae = np.where(there, ae + face * (e - np.roll(e, shift, axis)), ae)
    g6 = np.zeros((b, h, w), dtype=f)
    inner = (slice(None), slice(m, h - m), slice(m, w - m))
    g6[inner] = (f(2.0) / f(b * (h - 2 * m) * (w - 2 * m))) * ae[inner]
    flat, n, want = g6.ravel(), b * h * w, f(0.0)
    for c in range(256):
        run = f(0.0)
        for v in flat[n * c // 256:n * (c + 1) // 256]:
            run = f(run + v)
        want = f(want + run)
    assert g6.dtype == f and grad[co.OFF_B6] == want
