"""The RMSNorm that holds a row in one wave's registers gives the looping
kernel's bits: widths at the edges of 1024, 2048 and 4096 values and of a wave's
256, no delta, a delta and K-split partials, every output type. The looping
kernel takes the same aligned rows where the weights come as fp16 (of the same
values), and rows behind a 4-byte offset, whose squares it sums in another order
(held to a bound)."""

import pytest
import torch

from siliconfer_amd import _lib

pytestmark = pytest.mark.gpu


def _at(t, off):
    """A copy of t at a 16-byte boundary (off 0) or 4 bytes behind one."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("odt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("parts", [None, 0, 1, 2, 5, 8, 9])
@pytest.mark.parametrize("rows,H", [(1, 4), (3, 896), (2, 1020), (2, 1024), (5, 1028), (2, 2048), (3, 2052),
                                    (2, 4096), (1, 4100), (2, 1022)])
def test_same_bits(dev, rows, H, parts, odt):
    g = torch.Generator(device=dev).manual_seed(H + (parts or 0))
    x = torch.randn(rows, H, device=dev, generator=g)
    w16 = torch.randn(H, device=dev, generator=g).half()
    w = w16.float()
    d = torch.randn(max(parts or 1, 1), rows, H, device=dev, generator=g)
    lib, res = _lib.load(), []
    for off, weight in ((0, w), (0, w16), (1, w)):
        xv, wv, dv = _at(x, off), _at(weight, 0), _at(d, 0)
        out = torch.zeros(rows, H, dtype=odt, device=dev)
        if parts:
            rc = lib.sf_rmsnorm_partials(xv.data_ptr(), dv.data_ptr(), parts, wv.data_ptr(), _lib.dt(wv),
                                         out.data_ptr(), _lib.dt(out), rows, H, 1e-6, _lib.stream(xv))
        else:
            rc = lib.sf_rmsnorm(xv.data_ptr(), None if parts is None else dv.data_ptr(), wv.data_ptr(),
                                _lib.dt(wv), out.data_ptr(), _lib.dt(out), rows, H, 1e-6, _lib.stream(xv))
        assert rc == 0
        res.append((xv.clone(), out))
    x64 = x.double() + (0 if parts is None else d.double().sum(0))
    ref = x64 * torch.rsqrt((x64 * x64).mean(1, keepdim=True) + 1e-6) * w.double()
    for xs, out in res[1:]:
        assert torch.equal(res[0][0], xs)
    assert torch.equal(res[0][1], res[1][1])
    # the looping kernel sums a misaligned row's squares in another order: H * 2^-24 of the
    # sum, halved by the root, then three roundings and the output's own
    ulp = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.float32: 2.0**-24}[odt]
    bar = (H * 2.0**-25 + 8 * 2.0**-24 + ulp) * ref.abs() + (9 * 2.0**-24) * w.abs().double() * 8 + 2.0**-24
    for _, out in res:
        assert bool(((out.double() - ref).abs() <= bar).all())
