"""RoPE + append with four heads a workgroup (many rows) stores the bytes of the
same rows sent a few at a time (one head a workgroup), with head counts that do
and do not fill the last workgroup, from rows and from K-split partials."""

import pytest
import torch

from siliconfer_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("rows,H,KVH,D", [(512, 14, 2, 64), (700, 3, 2, 128), (300, 13, 1, 256), (4096, 1, 1, 62)])
def test_same_bytes(dev, rows, H, KVH, D, parts):
    assert rows * (H + 2 * KVH) >= 4096
    g = torch.Generator(device=dev).manual_seed(rows)
    W = (H + 2 * KVH) * D
    src = torch.randn(max(parts, 1), rows, W, device=dev, generator=g)
    ang = torch.rand(rows, D // 2, device=dev, generator=g) * 6
    cos, sin = ang.cos().contiguous(), ang.sin().contiguous()
    bias = torch.randn(W, device=dev, generator=g)
    lib, res = _lib.load(), []
    for step in (rows, 100):
        q = torch.zeros(rows, H, D, device=dev)
        kc = torch.zeros(KVH, rows, D, dtype=torch.int8, device=dev)
        vc, ks = kc.clone(), torch.zeros(KVH, rows, dtype=torch.float16, device=dev)
        vs = ks.clone()
        for r in range(0, rows, step):
            n = min(step, rows - r)
            assert step == rows or n * (H + 2 * KVH) < 4096
            x = src[:, r:r + n].contiguous()
            tail = (cos.data_ptr(), sin.data_ptr(), rows, q[r:].data_ptr(), _lib.SF_F32, kc.data_ptr(),
                    ks.data_ptr(), vc.data_ptr(), vs.data_ptr(), _lib.SF_F16, n, H, KVH, D, rows, None, r,
                    _lib.stream(q))
            rc = (lib.sf_rope_kv_append_partials(x.data_ptr(), parts, bias.data_ptr(), _lib.SF_F32, *tail)
                  if parts else lib.sf_rope_kv_append(x.data_ptr(), *tail))
            assert rc == 0
        res.append((q, kc, vc, ks, vs))
    for a, b in zip(*res):
        assert torch.equal(a, b)
