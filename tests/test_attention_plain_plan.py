"""CPU test of which plain-layout launches take the plain kernel and which the
generic one (chunks of 48 or 64 tokens with 4 or 8 query rows per kv head), through
the C ABI's workspace-size entry point: the generic kernel's plan has one unit of
split work per chunk and per 64 window tokens and aims at 2048 workgroups, the
plain kernel's keeps 3 chunks per wave or one workgroup per CU."""

import pytest

from intel_kivi_hybrid_amd import _native


def _splits(B, hg, D, G, Gv, chunks, window=100):
    rows = 1 if hg == 1 else 2 if hg == 2 else 4 if hg <= 4 else 8
    ws = _native.load().kivi_packed_decode_attention_workspace_size(
        B, 8 * hg, 8, D, G, Gv, chunks, window, 0)
    per = B * 8 * rows * (D + 2) * 4
    assert ws % per == 0
    return ws // per if ws else 1


def _generic(B, chunks, window=100):
    units = chunks + (window + 63) // 64
    s = max(1, min(-(-2048 // (B * 8)), -(-units // 4)))
    per = -(-units // s)
    return -(-units // per)


@pytest.mark.parametrize("B,hg,D,G,Gv,chunks,plain", [
    (4, 8, 96, 32, 32, 125, True),       # up to 32 tokens per chunk: always
    (4, 8, 96, 64, 32, 61, False),       # 8 rows, 64 tokens: 2 chunks per wave
    (1, 8, 96, 64, 32, 467, False),      # 3.6
    (16, 8, 96, 64, 32, 61, True),       # 7.6
    (16, 8, 96, 48, 32, 82, False),      # 48 tokens: never beyond the smallest
    (1, 8, 96, 64, 32, 4, True),
    (4, 4, 96, 64, 96, 61, True),        # 4 rows of 64 factors
    (4, 4, 80, 48, 16, 82, False),       # of 240 factors: 2.6 chunks per wave
    (1, 4, 80, 48, 16, 624, True),       # 4.9
    (1, 4, 80, 48, 16, 10, True),
    (4, 2, 48, 48, 16, 82, True),        # 1 and 2 rows: always
    (4, 1, 48, 48, 16, 82, True),
])
def test_which_kernel_takes_a_launch(B, hg, D, G, Gv, chunks, plain):
    splits = _splits(B, hg, D, G, Gv, chunks)
    if chunks > 12:                      # (tiny contexts: one split either way)
        assert (splits != _generic(B, chunks)) == plain


def test_every_cu_has_a_workgroup():
    """4 rows of 64 tokens per chunk: 32 pairs take 8 splits, 3 chunks per wave
    would leave 4."""
    assert _splits(4, 4, 96, 64, 96, 61) == 8
    assert _splits(4, 4, 96, 32, 96, 61) == 4
