"""CPU tests of the split plan of attention with more than 8 query rows per kv
head, through the C ABI's workspace-size entry point: S > 1 splits need batch *
q_len * q_heads * S * (head_dim + 2) fp32 of partials."""

import pytest

from intel_kivi_hybrid_amd import _native


def _splits(B, L, Hq, Hkv, D, G, chunks, window, hint):
    ws = _native.load().kivi_packed_attention_workspace_size(
        B, L, Hq, Hkv, D, G, G, chunks, window, hint)
    per = B * L * Hq * (D + 2) * 4
    assert ws % per == 0
    return ws // per if ws else 1


def test_a_callers_count_is_followed_while_the_partials_are_small():
    for hint in (2, 3, 8, 32):
        assert _splits(1, 5, 32, 8, 128, 32, 1024, 128, hint) == hint
    assert _splits(1, 512, 32, 8, 128, 32, 252, 640, 4) == 4


@pytest.mark.parametrize("B,L,Hq,Hkv,D,hint", [
    (1, 512, 32, 8, 128, 32), (1, 512, 32, 8, 128, 256), (8, 512, 32, 8, 128, 8),
    (4, 64, 16, 4, 256, 4096), (64, 40, 12, 12, 64, 64),
])
def test_partials_stay_below_64_mb(B, L, Hq, Hkv, D, hint):
    """(or what the decode kernel's launches of 8 rows, which take buffers off the
    wide loads' alignment, need with as many splits)"""
    ws = _native.load().kivi_packed_attention_workspace_size(
        B, L, Hq, Hkv, D, 32, 32, 4096, 640, hint)
    decode = B * Hkv * 8 * min(hint, 1024) * (D + 2) * 4
    assert ws <= max(64 << 20, decode)


@pytest.mark.parametrize("B,Hkv,hg,L,D", [
    (1, 1, 4, 512, 128), (1, 8, 4, 512, 128), (1, 8, 4, 5, 128), (16, 8, 4, 5, 128),
    (1, 32, 1, 512, 128), (1, 4, 4, 512, 256), (1, 12, 1, 512, 64), (8, 12, 1, 33, 64),
    (64, 8, 4, 512, 128),
])
def test_the_plans_own_count_is_not_cut(B, Hkv, hg, L, D):
    """One workgroup per CU (two where a workgroup holds at most 32 rows)."""
    rows = L * hg
    few = rows <= (64 if D == 64 else 32 if D == 128 else 16)
    block = (32 if rows > 16 and D <= 128 else 16) if few else \
        64 if D == 256 else 256 if rows > 128 else 128
    groups = B * Hkv * -(-rows // block)
    want = max(1, (512 if few else 256) // groups)
    got = _splits(B, L, Hkv * hg, Hkv, D, 32, 8192, 640, 0)
    assert want // 2 < got <= want
