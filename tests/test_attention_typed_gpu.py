"""Queries in the model's own type and strides (kivi_packed_attention_typed):
the same bits as the fp32 call on converted tensors, since queries widen exactly
and the output is rounded once, to nearest even, either way."""

import pytest
import torch

from tests.test_attention_rows_gpu import _store

CASES = [
    # B, Hq, Hkv, D, G, Gv, R, T, L, ring; rows per kv head at both kernels and
    # at one and several splits
    (1, 3, 1, 128, 32, 32, 64, 300, 3, "bf16"),        # 9 rows, one split
    (2, 8, 2, 128, 32, 32, 64, 2000, 5, "bf16"),       # 20 rows, splits
    (1, 11, 1, 64, 32, 32, 64, 500, 3, "f16"),         # 33 rows
    (1, 4, 2, 128, 64, 64, 128, 1300, 67, "f32"),      # 134 rows: the shared kernel
    (1, 2, 1, 256, 32, 256, 64, 400, 50, "bf16"),      # head_dim 256
    (64, 16, 4, 64, 32, 32, 64, 200, 20, "f16"),       # 80 rows, no split
    (1, 4, 2, 64, 32, 32, 64, 20, 5, "f32"),           # the window alone
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
def test_typed_queries_give_the_converted_call_bits(hip_device, case, dtype):
    from intel_kivi_hybrid_amd import _C
    B, Hq, Hkv, D, G, Gv, R, T, L, ring = case
    st, _, _ = _store(hip_device, B, Hkv, D, G, Gv, R, T, L, ring)
    g = torch.Generator().manual_seed(L + D)
    q = torch.randn(B, L, Hq + 1, D, generator=g).to("cuda", dtype)
    mask = torch.rand(B, T + L, generator=g) < 0.8
    mask[:, T] = True
    hidden = _C.hidden_positions(mask, q.device)
    start = torch.full((B,), min(7, T), dtype=torch.int32, device="cuda")
    token_major = q[:, :, 1:].transpose(1, 2)          # [B, Hq, L, D], as models hold it
    huge = token_major.clone()
    huge[0, 0, 0, 0] = 3.4e38 if dtype is not torch.float16 else float("inf")
    forms = [(token_major, {}), (token_major.contiguous(), {}),
             (token_major, {"kv_start": start}), (token_major, {"hidden": hidden}),
             (huge, {})]                               # (not finite as bf16)
    for x, kw in forms:
        assert _C.takes_typed_queries(x, st)
        got = _C.packed_attention_typed(x, st, **kw)
        want = _C.packed_attention(x.float(), st, **kw).to(dtype)
        assert got.dtype is dtype and got.shape == want.shape
        nan = got.isnan()
        assert torch.equal(nan, want.isnan())
        assert torch.equal(got[~nan], want[~nan])
    # what the loads cannot take goes the converted way
    pad = torch.zeros(B, Hq, L, D + 2, device="cuda", dtype=dtype)
    assert not _C.takes_typed_queries(pad[..., 1:D + 1], st)      # strides of 2 elements
    assert not _C.takes_typed_queries(token_major.double(), st)
    flat = torch.zeros(B * Hq * L * D + 1, device="cuda", dtype=dtype)[1:]
    assert not _C.takes_typed_queries(flat.view(B, Hq, L, D), st)
    assert not _C.takes_typed_queries(token_major[:, :, :1], st)


def test_typed_entry_refuses_before_any_launch():
    from intel_kivi_hybrid_amd import _native
    lib = _native.load()
    p = 4096

    def call(q=p, dt=1, sb=1024, q_len=3, heads=16, D=128):
        return lib.kivi_packed_attention_typed(
            q, dt, sb, 512, 128, q_len, 1, None, None, 0, p, p, p, p, p, p, p, p, 1, p, p,
            1 << 40, 1, heads, 4, D, 32, 32, 4, 2, 64, 0, 40, 1.0, 0, None)

    assert call(dt=3) == 1 and "q_dtype" in _native.last_error()
    assert call(q=p + 8) == 1 and "aligned" in _native.last_error()
    assert call(sb=1022) == 1 and "aligned" in _native.last_error()
    assert call(q_len=2) != 0 and "more than 8 rows" in _native.last_error()   # 8 rows
    assert call(D=96) != 0 and "more than 8 rows" in _native.last_error()      # plain layout
