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
