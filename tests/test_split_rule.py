"""The decode attention's default split count: unchanged up to one workgroup per
CU (256), and between one and two per CU above, never below 128 tokens a split
for the second."""

import pytest

from siliconfer_amd import _lib


@pytest.mark.parametrize("B,KVH", [(1, 1), (1, 2), (4, 2), (1, 8), (2, 8), (4, 8), (1, 32), (4, 32), (64, 32)])
def test_default_splits_over_batches(B, KVH):
    lib = _lib.load()
    for T in list(range(1, 700, 13)) + [1000, 2048, 2049, 4096, 8191, 16384, 100000]:
        base = 1 if T <= 160 else min(128, max(8, -(-T // (32 if T <= 2048 else 64))))
        s = lib.sf_attn_default_splits_d(B, KVH, T, 128)
        assert 1 <= s <= base
        if base * B * KVH <= 256:
            assert s == base
        else:
            assert s * B * KVH < 256 + B * KVH or (s * B * KVH <= 512 and s <= -(-T // 128)) or s == 1
            assert s * B * KVH >= min(256, base * B * KVH)
