"""CPU test of the split rule's exact fill at head_dim 128: where 512 / (B *
Hkv), 2 or 4, splits put two workgroups on every one of 256 CUs, they are taken
as soon as every wave keeps 9 chunks (6 with 8 query rows per kv head)."""

import pytest

from intel_kivi_hybrid_amd import _native


@pytest.mark.parametrize("B,Hq,n_chunks,S", [
    (16, 64, 95, 2), (16, 64, 96, 4),        # 8 rows: 4 splits from 6 chunks per wave
    (16, 32, 143, 2), (16, 32, 144, 4),      # 4 rows: from 9
    (32, 32, 71, 1), (32, 32, 72, 2),
    (64, 32, 252, 1),                        # one split already fills the chip
    (24, 32, 252, 2),                        # 512 / 192 is no whole number
    (8, 32, 432, 7), (8, 8, 288, 4),         # 8 splits: the count of >= 16 chunks per wave
    (8, 64, 384, 6), (4, 32, 864, 14),       # is as good or better
])
def test_splits_fill_the_chip(B, Hq, n_chunks, S):
    D, Hkv = 128, 8
    ws = _native.load().kivi_packed_decode_attention_workspace_size(
        B, Hq, Hkv, D, 32, 32, n_chunks, 128, 0)
    assert (ws // (B * Hq * (D + 2) * 4) if ws else 1) == S
