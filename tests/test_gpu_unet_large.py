"""The U-Net where element counts pass 2^31: a layer with that many weights,
and tensors with that many elements.  Indices into them take 64 bits."""
import numpy as np
import pytest

from hemelb_amd import warmstart as WS
from oracle import unet_oracle as U
from tests.test_gpu_unet import _case, _rel

pytestmark = pytest.mark.gpu


def test_forward_of_a_layer_of_2_31_weights():
    # 27 * 8928^2 weights in the coarsest level's second convolution.  Only 16
    # of its channels have non-zero weights, so the network computes what the
    # one of 16 channels does, to which the oracle is compared (with the
    # tolerance of test_gpu_unet.py: the same bfloat16 roundings).
    wide, side = 8928, 8
    narrow, chans = (16, 16, 16, 16), (16, 16, 16, wide)
    assert 27 * wide * wide >= 1 << 31
    _, p, x, _, _ = _case(side, 1, narrow, 31)
    p["e4b.w"] = p["e4b.w"] * np.float32(1024)   # so that the layer shows in the output
    net = WS.UNet(side, 1, 6, 4, chans)
    print(f"[unet] chans={chans} {net.device_bytes() / 2**30:.1f} GiB", flush=True)
    big = np.zeros(net.nparam, np.float32)
    q = WS.unpack(big, chans)             # views into `big`
    for k, a in p.items():
        if a.ndim == 1:
            q[k][:a.shape[0]] = a
        elif k == "d3a.w":                # input channels [upsampled, skip]
            q[k][:, :, :16], q[k][:, :, wide:] = a[:, :, :16], a[:, :, 16:]
        elif a.ndim == 3:
            q[k][:, :a.shape[1], :a.shape[2]] = a
        else:
            q[k][:] = a
    net.set_params(big)
    xp = np.concatenate([x, np.zeros(x.shape[:-1] + (10,), np.float32)], -1)
    pp = {k: a.astype(np.float64) for k, a in p.items()}
    out = U.forward(pp, xp, bf16=True)
    without = U.forward({**pp, "e4b.w": np.zeros_like(pp["e4b.w"])}, xp, bf16=True)
    assert _rel(without, out) > 0.1
    err = _rel(net.forward(x), out)
    assert err < 2e-2, err


def test_gradients_past_2_31_elements():
    # The concatenated gradient of the third level has 255 * 16^3 * 2096
    # elements.  The first and the last sample are the same crop, so a loss
    # over either has the same gradients: the same products, added in another
    # order in binary32 (runs of at most 2^26 terms in partial sums of partial
    # sums, nearly all of them zero: below 1e-4 of a tensor's norm).
    side, batch, chans = 64, 255, (16, 16, 16, 2080)
    assert batch * (side // 4) ** 3 * (chans[3] + chans[2]) >= 1 << 31
    net = WS.UNet(side, batch, 6, 4, chans)
    print(f"[unet] chans={chans} {net.device_bytes() / 2**30:.1f} GiB", flush=True)
    net.set_params(WS.init_params(chans, seed=32))
    rng = np.random.default_rng(33)
    x = np.zeros((batch, side, side, side, 6), np.float32)
    t = np.zeros((batch, side, side, side, 4), np.float32)
    x[0] = x[-1] = rng.standard_normal(x.shape[1:], np.float32)
    t[0] = t[-1] = rng.standard_normal(t.shape[1:], np.float32)
    mask = np.zeros((batch, side, side, side), np.uint8)
    y = net.forward(x)
    np.testing.assert_array_equal(y[0], y[-1])
    grads, losses = [], []
    for sample in (0, -1):
        mask[:] = 0
        mask[sample] = 1
        losses.append(net.backward(t, mask))
        grads.append(WS.unpack(net.grads(), chans))
    assert losses[0] > 0 and abs(losses[1] - losses[0]) <= 2e-5 * losses[0]
    errs = {k: _rel(grads[1][k], a) for k, a in grads[0].items()}
    print("[unet] relative differences", {k: f"{e:.1e}" for k, e in errs.items()}, flush=True)
    assert all(np.linalg.norm(a) > 0 for a in grads[0].values())
    assert max(errs.values()) < 1e-4, errs
