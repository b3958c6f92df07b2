"""sf_q4_matmul_group against the oracle's GEMM: column tiles of several weights
side by side (tails inside each weight, an output whose parts are not whole
16-byte pieces) and the SwiGLU tile (odd widths around its 64 columns, packed
and separate weights), one to four row blocks, one and two K groups, every
group size class and dtype."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import linear, primitives as P
from siliconfer_amd import _lib
from siliconfer_amd.kernels import Q4Weight
from siliconfer_amd.kernels.q4 import matmul_group
from siliconfer_amd.model.layers import MLP
from siliconfer_amd.model.q4_linear import Q4Linear

pytestmark = pytest.mark.gpu


def _weight(rng, N, K, g, asym):
    W = rng.normal(0, 0.02, (N, K)).astype(np.float32)
    if asym:
        return P.pack_weights_asym(W, g)
    (pk, s) = P.pack_weights_sym(W, g)
    return pk, s, None


def _ref(w, x, g):
    return linear.gemm(w[0], w[1].astype(np.float16).astype(np.float64),
                       x.float().cpu().numpy().astype(np.float64), g, zeros=w[2])


SHAPES = [  # M, Ns, K, g
    (17, (136, 8, 24), 96, 32), (33, (128, 128), 256, 64), (40, (130, 65, 7), 448, 64),
    (100, (4096, 1024, 1024), 768, 128), (333, (2056, 264, 264), 640, 128), (700, (896, 128, 128), 896, 64),
]


@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("xdtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,Ns,K,g", SHAPES)
def test_side_by_side(dev, M, Ns, K, g, xdtype, asym):
    rng = np.random.default_rng(M + K)
    parts = [_weight(rng, N, K, g, asym) for N in Ns]
    x = torch.as_tensor(rng.normal(0, 1, (M, K)).astype(np.float32)).to(dev).to(xdtype)
    b = [rng.normal(0, 0.1, N).astype(np.float32) if i != 1 else None for i, N in enumerate(Ns)]
    y = matmul_group(_lib.SF_GROUP_CONCAT, [Q4Weight(*p, g, device=dev) for p in parts], x,
                     [None if v is None else torch.as_tensor(v).to(dev) for v in b], out_dtype=torch.float32)
    ref = np.concatenate([_ref(p, x, g) + (0 if v is None else v) for p, v in zip(parts, b)], axis=1)
    y = y.double().cpu().numpy()
    assert y.shape == ref.shape
    # fp32 sums of exact products (fp32 activations drop at most 2^-17 of each)
    assert np.linalg.norm(y - ref) <= 2e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("xdtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,I,K,g", [(17, 64, 96, 32), (31, 63, 256, 64), (65, 130, 448, 64),
                                     (200, 1000, 640, 128), (512, 4864, 640, 64)])
def test_swiglu(dev, M, I, K, g, xdtype, asym, packed):
    rng = np.random.default_rng(M + I + K)
    gate, up = _weight(rng, I, K, g, asym), _weight(rng, I, K, g, asym)
    x = torch.as_tensor(rng.normal(0, 1, (M, K)).astype(np.float32)).to(dev).to(xdtype)
    if packed:
        both = [None if a is None else np.concatenate([a, c]) for a, c in zip(gate, up)]
        ws = [Q4Weight(*both, g, device=dev)]
    else:
        ws = [Q4Weight(*w, g, device=dev) for w in (gate, up)]
    y = matmul_group(_lib.SF_GROUP_SWIGLU, ws, x, out_dtype=torch.float32).double().cpu().numpy()
    G, U = _ref(gate, x, g), _ref(up, x, g)
    silu = G / (1 + np.exp(-G))
    # 2e-5 of each projection's norm, through |silu'| <= 1.1 and the product;
    # the fp32 exp, reciprocal and products add under 1e-6
    bar = 2e-5 * (1.1 * np.abs(U).max() * np.linalg.norm(G) + np.abs(silu).max() * np.linalg.norm(U))
    assert np.linalg.norm(y - silu * U) <= bar + 1e-6 * np.linalg.norm(silu * U)


def test_hooked_projection_is_called(dev):
    """A hook on a projection sees its call and may replace the output."""
    class Cfg:
        hidden_size, intermediate_size = 256, 320

    rng = np.random.default_rng(3)
    mlp = MLP(Cfg)
    for name, (n, k) in dict(gate_proj=(320, 256), up_proj=(320, 256), down_proj=(256, 320)).items():
        setattr(mlp, name, Q4Linear(*_weight(rng, n, k, 64, False), group_size=64, device=dev))
    x = torch.as_tensor(rng.normal(0, 1, (1, 40, 256)).astype(np.float32)).to(dev)
    plain = mlp(x)
    seen = []
    h = mlp.up_proj.register_forward_hook(lambda m, a, out: seen.append(out.shape) or out * 2)
    twice = mlp(x)
    h.remove()
    assert seen == [torch.Size([1, 40, 320])]
    # each route: 2e-5 of the norm a projection, three in a row, the SwiGLU's product with
    # max / rms factors of about 4 for normal draws: under 2.5e-4 each
    assert float((twice - 2 * plain).norm()) <= 5e-4 * float(2 * plain.norm())


def test_refused_forms(dev):
    lib = _lib.load()
    Ns = (ctypes.c_int * 2)(64, 72)
    assert lib.sf_q4_matmul_group_supported(_lib.SF_GROUP_SWIGLU, 2, Ns, 64, 256, 64, _lib.SF_F16, None) == 0
    assert lib.sf_q4_matmul_group_supported(_lib.SF_GROUP_CONCAT, 2, Ns, 16, 256, 64, _lib.SF_F16, None) == 0
    assert lib.sf_q4_matmul_group_supported(_lib.SF_GROUP_CONCAT, 2, Ns, 64, 256, 48, _lib.SF_F16, None) == 0
    assert lib.sf_q4_matmul_group_supported(_lib.SF_GROUP_CONCAT, 2, Ns, 64, 256, 64, _lib.SF_F16, None) == 1
    # a weight that splits K by itself keeps its shorter sums
    Ns = (ctypes.c_int * 2)(4096, 1024)
    assert lib.sf_q4_matmul_group_supported(_lib.SF_GROUP_CONCAT, 2, Ns, 300, 4096, 64, _lib.SF_F16, None) == 0
