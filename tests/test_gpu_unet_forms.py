"""The U-Net where its launch rules choose otherwise than in the other tests.
The oracle and its tolerances are those of test_gpu_unet.py (bfloat16 against
binary64 with the same roundings)."""
import numpy as np
import pytest

from hemelb_amd import warmstart as WS
from oracle import unet_oracle as U
from tests.test_gpu_unet import _case, _rel

pytestmark = pytest.mark.gpu

CASES = [
    (8, 300, (16, 32, 64, 128)),    # many small samples: no boxes from 4^3 down
]


@pytest.mark.parametrize("side,batch,chans", CASES)
def test_forward_and_gradients_match_oracle(side, batch, chans):
    print(f"[unet] side={side} batch={batch} chans={chans}", flush=True)
    v, p, x, t, mask = _case(side, batch, chans, 5 * side + batch)
    net = WS.UNet(side, batch, 6, 4, chans)
    net.set_params(v)
    y = net.forward(x)
    xp = np.concatenate([x, np.zeros(x.shape[:-1] + (10,), np.float32)], -1)
    pp = {k: a.astype(np.float64) for k, a in p.items()}
    out, acts = U.forward(pp, xp, bf16=True, keep=True)
    err = _rel(y, out)
    assert err < 2e-2, err
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
