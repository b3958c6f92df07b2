"""Decode attention on MFMA over V scales from tiny to beyond what fp16 weights
times 2^10 hold, one split and several, garbage scales past the length, against
float64. q and the weights keep 22 bits as two fp16 halves; a weight's low half
ends at 2^-25, over the 2^10 where a wave runs more than one tile (n_splits 1
and 2 over 1200 tokens do): 2e-6 + sqrt(1200) * 2^-35 * 32 / scale (2^-25
without) bounds the error, for weights of sqrt(sum p^2) >= 1/32."""

import pytest
import torch

from siliconfer_amd.kernels.attention import attention_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_splits", [1, 2, 37])
@pytest.mark.parametrize("H,KVH,D", [(14, 2, 64), (32, 8, 128)])
@pytest.mark.parametrize("vscale", [1e-5, 0.02, 40.0, 3000.0])
def test_v_scale_range(dev, vscale, H, KVH, D, n_splits):
    out, ref = run(dev, vscale, H, KVH, D, n_splits)
    assert float((out - ref).norm() / ref.norm()) < 2e-6 + (3.3e-8 if n_splits <= 2 else 3.3e-5) / vscale


@pytest.mark.parametrize("n_splits", [1, 2])
@pytest.mark.parametrize("H,KVH,D", [(14, 2, 64), (32, 8, 128)])
@pytest.mark.parametrize("at", [3, 700, 1186])
@pytest.mark.parametrize("value", [1e9, 1e38])
def test_faint_large_v_scale(dev, H, KVH, D, n_splits, at, value):
    """One large fp32 V scale whose token weighs next to nothing for all heads
    but each kv head's first: the others keep their bits. Its score is -2 * 127 *
    0.022 * sqrt(D) = -45 (D = 64) or -63 for them, give or take 127 * 0.022 *
    0.7 = 2 (a weight times 1e9 under 1e-5), and as much above zero for the
    first. 1e38 comes with a score three times as low, a weight that is 0, and a
    factor of 2^-2 that keeps the scale itself in fp32: 2^-25 over that."""
    out, ref = run(dev, 0.02, H, KVH, D, n_splits, (at, value))
    G = H // KVH
    for h in range(H):
        o, r = out[:, h], ref[:, h]
        if h % G == 0 and value > 1e30:  # weights that leave fp16 at every factor
            assert not bool(torch.isfinite(o).any())
        else:
            assert float((o - r).norm() / r.norm()) < 2e-6 + (3.3e-8 if value < 1e30 else 4 * 3.3e-5) / 0.02


def run(dev, vscale, H, KVH, D, n_splits, spike=None):
    g = torch.Generator(device=dev)
    g.manual_seed(D + n_splits)
    B, T, cap = 2, 1200 - 13, 1200
    kc = torch.randint(-128, 128, (B, KVH, cap, D), generator=g, device=dev).to(torch.int8)
    vc = torch.randint(-128, 128, (B, KVH, cap, D), generator=g, device=dev).to(torch.int8)
    ks = 0.01 + 0.01 * torch.rand(B, KVH, cap, generator=g, device=dev)
    vs = vscale * (0.5 + torch.rand(B, KVH, cap, generator=g, device=dev))
    ks[:, :, T:], vs[:, :, T:] = float("nan"), float("inf")
    q = 0.7 * torch.randn(B, H, D, generator=g, device=dev)
    if spike is not None:  # (token, its V scale): scored low, but by each kv head's first query
        q += 2
        q[:, ::H // KVH] -= 4
        kc[:, :, spike[0]], vs[:, :, spike[0]] = -127, spike[1]
        ks[:, :, spike[0]] = 0.022 if spike[1] < 1e30 else 0.066
    out = attention_decode(q, kc, ks, vc, vs, T=T, n_splits=n_splits).double()
    ref = torch.empty(B, H, D, dtype=torch.float64, device=dev)
    for b in range(B):
        for h in range(H):
            j = h // (H // KVH)
            s = (kc[b, j, :T].double() * ks[b, j, :T, None].double()) @ q[b, h].double() * D ** -0.5
            ref[b, h] = torch.softmax(s, 0) @ (vc[b, j, :T].double() * vs[b, j, :T, None].double())
    return out, ref
