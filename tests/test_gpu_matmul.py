"""sf_q4_matmul (every kernel it chooses between) against the oracle's GEMM at
the edges of its tiles: one row (bf16 with zero-points at long K goes to the rows
kernel), row counts around the GEMV's 8 and 16, the 32-row blocks and one to
four of them per tile, columns around the 128-wide tiles, K of one 32-group, of an odd number of 64-k steps and of several K splits, and
one and two K groups of waves. fp32 sums of exact products: the bar is 2e-5 of
the result's norm (fp32 activations drop at most 2^-17 of each)."""

import numpy as np
import pytest
import torch

from oracle import linear, primitives as P
from siliconfer_amd import _lib
from siliconfer_amd.kernels import Q4Weight

pytestmark = pytest.mark.gpu

SHAPES = [  # M, N, K, g
    (1, 200, 12288, 64), (1, 4096, 11008, 64), (2, 136, 11008, 64),
    (7, 130, 128, 64), (8, 264, 12288, 64), (9, 1000, 4224, 128), (16, 257, 8192, 64),
    (17, 128, 32, 32), (31, 127, 96, 32), (32, 129, 64, 64), (33, 896, 896, 64),
    (64, 1024, 4096, 128), (65, 300, 320, 64), (95, 2500, 1152, 128), (96, 4864, 896, 64),
    (97, 136, 2048, 256), (128, 5000, 640, 128), (200, 11008, 1024, 64), (333, 2056, 1984, 64),
    (512, 4864, 448, 64), (700, 12000, 256, 128),
]


@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("xdtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,g", SHAPES)
def test_matmul_tiles(dev, M, N, K, g, xdtype, asym):
    rng = np.random.default_rng(M * 7 + N + K)
    W = rng.normal(0, 0.02, (N, K)).astype(np.float32)
    if asym:
        pk, s, z = P.pack_weights_asym(W, g)
    else:
        (pk, s), z = P.pack_weights_sym(W, g), None
    w = Q4Weight(pk, s, z, g, device=dev)
    x = torch.as_tensor(rng.normal(0, 1, (M, K)).astype(np.float32)).to(dev).to(xdtype)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    y = w.matmul(x, out_dtype=torch.float32, bias=torch.as_tensor(b).to(dev)).double().cpu().numpy()
    s16 = s.astype(np.float16).astype(np.float64)
    ref = linear.gemm(pk, s16, x.float().cpu().numpy().astype(np.float64), g, zeros=z) + b
    assert np.linalg.norm(y - ref) <= 2e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("M,N,K,g,xdtype", [
    (3, 4096, 4096, 128, torch.float32), (8, 4096, 4096, 64, torch.float32), (1, 130, 12288, 64, torch.bfloat16),
    (8, 264, 12288, 64, torch.bfloat16), (9, 1000, 1152, 128, torch.float32), (12, 300, 4224, 64, torch.float16),
    (17, 129, 320, 32, torch.bfloat16), (40, 257, 1024, 64, torch.float16), (40, 256, 1024, 64, torch.float32),
    (11, 72, 336, 48, torch.float16)])
def test_matmul_residual(dev, M, N, K, g, xdtype):
    """bias == out_f32: every row adds its own previous values, whatever the shape's
    route without it (rows kernel, K splits, VALU kernel)."""
    rng = np.random.default_rng(M + N + K)
    pk, s, z = P.pack_weights_asym(rng.normal(0, 0.02, (N, K)).astype(np.float32), g)
    w = Q4Weight(pk, s, z, g, device=dev)
    x = torch.as_tensor(rng.normal(0, 1, (M, K)).astype(np.float32)).to(dev).to(xdtype)
    h = rng.normal(0, 3, (M, N)).astype(np.float32)
    y = torch.as_tensor(h).to(dev)
    w.matmul(x, bias=y, out_f32=y)
    ref = linear.gemm(pk, s.astype(np.float16).astype(np.float64), x.float().cpu().numpy().astype(np.float64), g,
                      zeros=z) + h
    assert np.linalg.norm(y.double().cpu().numpy() - ref) <= 2e-5 * np.linalg.norm(ref)


def test_matmul_workspace_is_checked(dev):
    lib = _lib.load()
    M, N, K, g = 40, 256, 1024, 64
    pk, s = P.pack_weights_sym(np.ones((N, K), np.float32), g)
    w = Q4Weight(pk, s, None, g, device=dev)
    x = torch.zeros(M, K, device=dev)
    y = torch.full((M, N), 7.0, device=dev)
    need = lib.sf_q4_matmul_workspace_bytes(M, N, K, g, _lib.SF_F32)
    assert need >= M * K * 4  # the halves of fp32 activations
    rc = lib.sf_q4_matmul(w.blob.data_ptr(), x.data_ptr(), _lib.SF_F32, y.data_ptr(), _lib.SF_F32, None,
                          None, 0, M, N, K, g, 0, None, 0, _lib.stream(x))
    assert rc == -1 and "workspace too small" in _lib.last_error()
    torch.cuda.synchronize()
    assert bool((y == 7.0).all())
