"""Causal prefill attention on 32-row workgroups (prompts of at least one such
workgroup per CU) against a float64 evaluation of the same codes and scales:
row counts around the 32-row blocks and 32-key tiles, with and without a cached
prefix, both head dims, fp16 / fp32 scales, NaN scales behind the cached length,
and V scales from tiny to beyond what fp16 weights times 2^10 would hold, one
huge or infinite among ordinary ones included: only the rows that see it may
change. q and the weights keep 22 bits (two fp16 halves): the bar is 2e-6 of the
norm."""

import numpy as np
import pytest
import torch

from siliconfer_amd import _lib

pytestmark = pytest.mark.gpu


def run(dev, T, T0, H, KVH, D, qdt, sdt, odt, vscale, dev_pos=False, spike=None, faint=False):
    g = torch.Generator(device=dev)
    g.manual_seed(T * 31 + T0 + D)
    n, cap = T0 + T, T0 + T + 3
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    kc = torch.randint(-128, 128, (KVH, cap, D), generator=g, device=dev).to(torch.int8)
    vc = torch.randint(-128, 128, (KVH, cap, D), generator=g, device=dev).to(torch.int8)
    ks = (0.01 + 0.01 * torch.rand(KVH, cap, generator=g, device=dev)).to(sdt)
    vs = (vscale * (0.5 + torch.rand(KVH, cap, generator=g, device=dev))).to(sdt)
    ks[:, n:], vs[:, n:] = float("nan"), float("nan")  # never-written rows
    q = 0.7 * r(T, H, D)
    if spike is not None:  # (key, its V scale); faint: a key that every query scores low
        vs[:, spike[0]] = spike[1]
        if faint:
            q += 2
            kc[:, spike[0]], ks[:, spike[0]] = -127, 0.022
    q = q.to(qdt)
    out = torch.full((T, H, D), float("nan"), dtype=odt, device=dev)
    st = _lib.stream(q)
    lib = _lib.load()
    args = (q.data_ptr(), _lib.dt(q), kc.data_ptr(), ks.data_ptr(), vc.data_ptr(), vs.data_ptr(), _lib.dt(ks),
            out.data_ptr(), _lib.dt(out))
    if dev_pos:
        pos = torch.tensor([T0], dtype=torch.int32, device=dev)
        _lib.check(lib.sf_attn_prefill_i8kv_dev(*args, None, 0, T, H, KVH, pos.data_ptr(), cap, cap, D,
                                                D ** -0.5, 1, st), "prefill_dev")
    else:
        _lib.check(lib.sf_attn_prefill_i8kv(*args, T, H, KVH, T0, cap, D, D ** -0.5, st), "prefill")
    k = kc[:, :n].double() * ks[:, :n, None].double()
    v = vc[:, :n].double() * vs[:, :n, None].double()
    mask = torch.arange(n, device=dev)[None, :] > torch.arange(T, device=dev)[:, None] + T0
    ref = torch.empty(T, H, D, dtype=torch.float64, device=dev)
    for h in range(H):
        s = q[:, h].double() @ k[h // (H // KVH)].t().contiguous() * D ** -0.5
        ref[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ v[h // (H // KVH)]
    return out.double(), ref


@pytest.mark.parametrize("T,T0,H,KVH,D,qdt,sdt", [
    (256, 0, 32, 8, 128, torch.float32, torch.float16),
    (257, 31, 32, 8, 128, torch.float16, torch.float16),
    (300, 33, 32, 8, 128, torch.bfloat16, torch.float32),
    (271, 1, 32, 32, 128, torch.float32, torch.float32),
    (600, 0, 14, 2, 64, torch.float16, torch.float16),
    (601, 95, 14, 2, 64, torch.float32, torch.float16),
    (1023, 64, 8, 8, 64, torch.bfloat16, torch.float16),
])
@pytest.mark.parametrize("dev_pos", [False, True])
def test_rows_against_float64(dev, T, T0, H, KVH, D, qdt, sdt, dev_pos):
    assert (T * (H // KVH) + 31) // 32 * KVH >= 256
    out, ref = run(dev, T, T0, H, KVH, D, qdt, sdt, torch.float32, 0.02, dev_pos)
    assert float((out - ref).norm() / ref.norm()) < 2e-6


@pytest.mark.parametrize("vscale", [1e-5, 0.5, 40.0, 3000.0])
@pytest.mark.parametrize("odt", [torch.float16, torch.bfloat16, torch.float32])
def test_rows_v_scale_range(dev, vscale, odt):
    """V scales whose weights times 2^10 leave fp16 shrink the factor instead."""
    out, ref = run(dev, 260, 0, 32, 8, 128, torch.float32, torch.float32, odt, vscale)
    if odt == torch.float16 and vscale > 100:  # fp16 results overflow as the values do
        ok = ref.abs() < 6e4
        out, ref = out[ok], ref[ok]
    # the output's own rounding (fp16 results near 1e-4 are subnormal), and each
    # weight's low half: half a subnormal step 2^-25 over the 2^10, random over up
    # to 260 keys, against a result of vscale * |code| * sqrt(sum p^2 >= 1 / 256):
    # sqrt(260) * 2^-35 * 16 / vscale < 8e-9 / vscale
    tol = {torch.float32: 4e-6, torch.float16: 2e-2 if vscale < 1e-3 else 1e-3, torch.bfloat16: 4e-3}[odt]
    tol += 8e-9 / vscale
    assert float((out - ref).norm() / ref.norm()) < tol


GEO = [(260, 0, 32, 8, 128), (601, 95, 14, 2, 64)]


@pytest.mark.parametrize("sdt,value", [(torch.float32, float("inf")), (torch.float16, float("inf")),
                                       (torch.float32, 1e9), (torch.float32, 1e38)])
@pytest.mark.parametrize("at", [0, 5, 31, 77, 150, 255])
@pytest.mark.parametrize("T,T0,H,KVH,D", GEO)
def test_rows_before_a_large_v_scale(dev, T, T0, H, KVH, D, at, sdt, value):
    """Rows that do not see the key keep their bits; rows that do meet the bar, or
    are not finite where the key's weights leave fp16 at every factor (2^10..2^-20)."""
    args = (dev, T, T0, H, KVH, D, torch.float32, sdt, torch.float32, 0.02)
    plain, _ = run(*args)
    out, ref = run(*args, spike=(T0 + at, value))
    assert torch.equal(out[:at], plain[:at])
    if value > 1e30:
        assert not bool(torch.isfinite(out[at:]).any())
    else:
        assert float((out[at:] - ref[at:]).norm() / ref[at:].norm()) < 4e-6


@pytest.mark.parametrize("T,T0,H,KVH,D", GEO)
def test_rows_faint_large_v_scale(dev, T, T0, H, KVH, D):
    """A 1e9 V scale whose key weighs next to nothing takes no bits from the
    other keys. Its score is -2 * 127 * 0.022 * sqrt(D) = -45 (D = 64) or -63, give
    or take 127 * 0.022 * 0.7 = 2: its weight times 1e9 stays under 1e-5."""
    out, ref = run(dev, T, T0, H, KVH, D, torch.float32, torch.float32, torch.float32, 0.02,
                   spike=(T0 + 40, 1e9), faint=True)
    assert float((out[41:] - ref[41:]).norm() / ref[41:].norm()) < 2e-6
