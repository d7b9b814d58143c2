"""The U-Net at sizes where its kernels' tiles, boxes and channel groups can go
wrong: widths that are no multiple of the 16- or 8-wide boxes, levels smaller
than a box, forms of the LDS convolution (groups of 16 channels, large and
small boxes, K in one slice and in several; the others in
test_gpu_unet_forms.py) and the channel counts that have none.  The oracle and its tolerances are those of test_gpu_unet.py
(bfloat16 against binary64 with the same roundings)."""
import numpy as np
import pytest

from hemelb_amd import warmstart as WS
from oracle import unet_oracle as U
from tests.test_gpu_unet import _case, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,batch,chans", [
    (24, 2, (16, 96, 128, 64)),     # 24, 12, 6, 3; 6, 8 and 12 groups; 7 and 14 have no form
    (40, 1, (16, 32, 32, 48)),      # 40, 20, 10, 5; 5 groups have no form
    (56, 1, (32, 16, 16, 16)),      # large 8-wide boxes, 3 groups into 2 tiles
    (56, 1, (16, 32, 16, 16)),      # large 8-wide boxes, 1 group into 1 and 3 tiles
    (64, 1, (32, 32, 16, 16)),      # large 16-wide boxes, 2 and 4 groups into 2 and 4 tiles
])
def test_forward_and_gradients_match_oracle(side, batch, chans):
    print(f"[unet] side={side} batch={batch} chans={chans}", flush=True)
    v, p, x, t, mask = _case(side, batch, chans, 3 * side + batch)
    net = WS.UNet(side, batch, 6, 4, chans)
    net.set_params(v)
    y = net.forward(x)
    xp = np.concatenate([x, np.zeros(x.shape[:-1] + (10,), np.float32)], -1)
    pp = {k: a.astype(np.float64) for k, a in p.items()}
    out, acts = U.forward(pp, xp, bf16=True, keep=True)
    assert _rel(y, out) < 2e-2, _rel(y, out)
    wts = np.array([1.0, 1.0, 1.0, 0.5])
    loss = net.backward(t, mask, wts)
    l_o, dout = U.loss_and_grad_out(y.astype(np.float64), t, mask, wts)
    assert abs(loss - l_o) <= 1e-4 * l_o
    g_o = U.backward(pp, acts, dout, bf16=True)
    g = WS.unpack(net.grads(), chans)
    worst = {name: _rel(g[name], g_o[name]) for name in g_o}
    print("[unet] relative gradient errors", {k: round(e, 4) for k, e in worst.items()},
          flush=True)
    assert max(worst.values()) < 5e-2, worst


def test_forward_of_the_smallest_crop():
    # levels of 8, 4, 2 and 1: with two positions at the coarsest level a
    # single ReLU that flips on a rounding moves its gradients by tens of per
    # cent, so only the output is compared
    side, batch, chans = 8, 2, (16, 32, 64, 128)
    v, p, x, _, _ = _case(side, batch, chans, 26)
    net = WS.UNet(side, batch, 6, 4, chans)
    net.set_params(v)
    xp = np.concatenate([x, np.zeros(x.shape[:-1] + (10,), np.float32)], -1)
    out = U.forward({k: a.astype(np.float64) for k, a in p.items()}, xp, bf16=True)
    out = out[0] if isinstance(out, tuple) else out
    assert _rel(net.forward(x), out) < 2e-2
