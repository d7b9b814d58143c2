"""The U-Net where its launch rules choose otherwise than in the other tests:
with those, every form of the LDS convolution runs, and each that the default
network reaches in the way it reaches it, K in one slice or in several
(test_unet_plan.py checks this against the rules).
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
    # medium boxes, 8 wide: 20^3 and 24^3 positions a sample
    (40, 5, (16, 32, 64, 128)),
    (48, 5, (16, 32, 64, 16)),
    # medium boxes, 16 wide
    (32, 2, (16, 32, 64, 128)),
    (64, 2, (16, 32, 16, 16)),
]

# Networks whose gradients are too ill-conditioned for a tolerance of 5e-2: with
# few positions on the coarse levels, rounding the oracle's own sums to
# binary32 flips ReLUs and moves its gradients by 2 to 5 per cent (by 0.3 to
# 1.6 in the networks above), so only the output is compared.
OUTPUT_CASES = [
    (24, 5, (16, 32, 64, 128)),     # 24^3: medium 8-wide boxes, 1 and 3 groups
    (56, 1, (16, 16, 16, 16)),      # large 8-wide boxes, 2 groups into 1 tile
    (24, 2, (64, 64, 16, 16)),      # many positions, 4 and 8 groups, 8 wide
    (32, 1, (64, 64, 16, 16)),      # the same, 16 wide
]


def forward(side, batch, chans):
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
    return net, y, t, mask, pp, acts


@pytest.mark.parametrize("side,batch,chans", OUTPUT_CASES)
def test_forward_matches_oracle(side, batch, chans):
    forward(side, batch, chans)


@pytest.mark.parametrize("side,batch,chans", CASES)
def test_forward_and_gradients_match_oracle(side, batch, chans):
    net, y, t, mask, pp, acts = forward(side, batch, chans)
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
