"""GPU parity of attention with more query rows per kv head than one decode
launch takes (q_len * Hq / Hkv > 8, matrix-core stores): the kernels that
dequantise each 32 tokens once for all rows.

Rows per kv head sit at the edges of the row tiles (16), of the two kernels (16,
32 or 64 by head_dim) and of the workgroups' row blocks (64, 128, 256); contexts end inside a 32-token
unit, lie wholly in the window, and split.  Against float64 attention over the
oracle's dequantised history, elementwise, with the bound that the arithmetic
gives.  Weights and packed values (their offset from the middle of their group's
range, at most 1.5 scales and so no more than the largest magnitude in the group)
are split into two bf16 pieces each (2^-18 relative) and their lo*lo product is
dropped (2^-18): 3 * 2^-18 of sum_t p_t |v_t|, where the data is of zero mean.
Keys carry three pieces; a score is then a fp32 sum of 6 D/32 matrix products
(three-piece queries), off by at most 6 D/32 * 2^-24 of sum_d |q_d k_d| *
scale, which moves a weight and the normaliser by as much each.
"""

import numpy as np
import pytest
import torch

from oracle.attention import decode_attention, prefix_attention
from tests.kv_helpers import make_kv, oracle_history, rel_err

pytestmark = pytest.mark.gpu

def _store(hip_device, B, Hkv, D, G, Gv, R, T, L, ring, v_offset=0.0):
    from intel_kivi_hybrid_amd.store import PackedKVStore
    dt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[ring]
    k, v = make_kv(B, Hkv, T + L, D, seed=T + L + D)
    k, v = k.to(dt).float(), (v + v_offset).to(dt).float()
    st = PackedKVStore(B, Hkv, D, G, R + L, "cuda:0", group_size_v=Gv, residual_dtype=dt,
                       chunk_capacity=T // G + 1)
    st.extend(k[:, :, :T].to("cuda", dt), v[:, :, :T].to("cuda", dt), flush_at=R)
    st.append(k[:, :, T:].to("cuda", dt), v[:, :, T:].to("cuda", dt))
    return st, k, v


def _bound(q, kh, kr):
    """The bound above for queries [B, L, Hq, D]."""
    B, L, Hq, D = q.shape
    keys = np.abs(np.concatenate([kh, kr], 2))
    qa = np.abs(q).reshape(B, L, keys.shape[1], -1, D)
    smax = max(float((qa[b, :, h].reshape(-1, D) @ keys[b, h].T).max())
               for b in range(B) for h in range(keys.shape[1])) * D ** -0.5
    return 3 * 2.0 ** -18 + 2 * (6 * D / 32) * 2.0 ** -24 * smax


def _check(out, q, st, k, v, G, Gv, **mask):
    kh, vh = oracle_history(k, v, st.n_chunks, G, Gv)
    q0 = st.n_chunks * G
    qn, kr, vr = q.transpose(1, 2).numpy(), k[:, :, q0:].numpy(), v[:, :, q0:].numpy()
    ref = prefix_attention(qn, kh, vh, kr, vr, **mask)
    size = prefix_attention(qn, kh, np.abs(vh), kr, np.abs(vr), **mask)
    bound = _bound(qn, kh, kr)
    err = np.abs(out.cpu().numpy().astype(np.float64) - ref) / np.maximum(size, 1e-30)
    print(f"[rows]   largest error {err.max():.2e} of sum p|v| (bound {bound:.2e})", flush=True)
    assert err.max() <= bound


CASES = [
    # B, Hq, Hkv, D, G, Gv, R, T, L, splits, ring, bf16 queries
    (1, 3, 1, 128, 32, 32, 64, 300, 3, 0, "f32", False),      # 9 rows, 3 query pieces
    (2, 4, 1, 128, 32, 32, 64, 777, 4, 0, "bf16", True),      # 16 rows: one tile
    (1, 17, 1, 64, 32, 32, 64, 333, 2, 3, "f16", True),       # 34 rows, 3 splits
    (1, 8, 1, 128, 32, 32, 64, 500, 4, 0, "f32", False),      # 32 rows
    (1, 11, 1, 128, 32, 32, 64, 500, 3, 2, "bf16", True),     # 33 rows
    (1, 4, 2, 128, 64, 64, 128, 1300, 32, 0, "f32", True),    # 64 rows, G = 64
    (1, 13, 1, 128, 32, 128, 64, 500, 5, 0, "bf16", False),   # 65 rows, one value group
    (1, 8, 2, 256, 64, 128, 128, 700, 4, 2, "f32", False),    # head_dim 256, 16 rows
    (1, 17, 1, 256, 32, 256, 64, 400, 2, 0, "f16", False),    # head_dim 256, 34 rows
    (1, 2, 1, 256, 32, 32, 64, 400, 50, 0, "bf16", True),     # head_dim 256, 100 rows
    (1, 4, 1, 128, 32, 32, 128, 2100, 33, 0, "bf16", True),   # 132 rows: two row tiles
    (2, 8, 4, 64, 64, 32, 64, 1000, 129, 2, "f16", False),    # 258 rows: two row blocks
    (1, 2, 2, 128, 32, 32, 128, 40, 300, 0, "f32", True),     # no chunk yet: the window alone
    (1, 4, 2, 64, 32, 32, 64, 20, 5, 0, "bf16", False),       # the same, few rows
]


@pytest.mark.parametrize("B,Hq,Hkv,D,G,Gv,R,T,L,splits,ring,half_q", CASES)
def test_rows_match_oracle(hip_device, B, Hq, Hkv, D, G, Gv, R, T, L, splits, ring, half_q):
    print(f"[rows] B={B} Hq={Hq} Hkv={Hkv} D={D} G={G} Gv={Gv} R={R} T={T} L={L} splits={splits} "
          f"{ring} half_q={half_q}", flush=True)
    st, k, v = _store(hip_device, B, Hkv, D, G, Gv, R, T, L, ring)
    g = torch.Generator().manual_seed(L + D)
    q = torch.randn(B, Hq, L, D, generator=g)
    if half_q:
        q = q.bfloat16().float()
    out = st.attention(q.cuda(), num_splits=splits)
    _check(out, q, st, k, v, G, Gv)
    assert torch.equal(out, st.attention(q.cuda(), num_splits=splits))
    # padding: a leading run, then holes (both kernels' masks, window included)
    total = st.quantized_tokens + st.res_len
    start = [min(37 * (b + 1), total - L) for b in range(B)]
    out = st.attention(q.cuda(), num_splits=splits, kv_start=start)
    _check(out, q, st, k, v, G, Gv, kv_start=np.array(start))
    vis = torch.rand(B, total, generator=g) >= 0.2
    vis[:, 0] = True
    out = st.attention(q.cuda(), num_splits=splits, key_mask=vis)
    _check(out, q, st, k, v, G, Gv, visible=vis.numpy())


def test_unaligned_queries(hip_device):
    """Queries and outputs off the 16-byte alignment of the wide loads."""
    B, Hq, L, D = 1, 8, 6, 128
    st, k, v = _store(hip_device, B, 2, D, 32, 32, 64, 300, L, "f32")
    q = torch.randn(B, L, Hq, D, generator=torch.Generator().manual_seed(3))
    base = torch.empty(q.numel() + 1, device="cuda")
    base[1:] = q.flatten().cuda()
    out = torch.empty(q.numel() + 1, device="cuda")[1:].view(B, L, Hq, D)
    st.attention(base[1:].view(B, L, Hq, D).transpose(1, 2), out=out)
    _check(out, q.transpose(1, 2), st, k, v, 32, 32)


@pytest.mark.parametrize("Hq,Hkv,D,G,Gv,T,L,splits", [
    (8, 1, 128, 32, 32, 500, 2, 0),          # 16 rows
    (24, 2, 64, 32, 32, 300, 2, 2),          # 12 heads: groups of 8 and 4
    (3, 1, 128, 64, 128, 700, 5, 0),         # 2 tokens per launch, 2 padding rows
    (4, 1, 256, 64, 128, 500, 3, 0),         # at most 4 rows per launch
])
def test_unaligned_queries_take_the_decode_launches(hip_device, Hq, Hkv, D, G, Gv, T, L, splits):
    """The decode kernel's launches of up to 8 rows, which buffers off the wide
    loads' alignment take, causal and not."""
    print(f"[rows] decode launches: Hq={Hq} Hkv={Hkv} D={D} G={G} T={T} L={L}", flush=True)
    st, k, v = _store(hip_device, 2, Hkv, D, G, Gv, 64, T, L, "f32")
    q = torch.randn(2, L, Hq, D, generator=torch.Generator().manual_seed(3)) * D ** -0.5
    base = torch.empty(q.numel() + 1, device="cuda")
    base[1:] = q.flatten().cuda()
    kh, vh = oracle_history(k, v, st.n_chunks, G, Gv)
    q0 = st.n_chunks * G
    kr, vr = k[:, :, q0:].numpy(), v[:, :, q0:].numpy()
    for causal in (True, False):
        out = torch.empty(q.numel() + 1, device="cuda")[1:].view(2, L, Hq, D)
        st.attention(base[1:].view(2, L, Hq, D).transpose(1, 2), out=out, causal=causal,
                     num_splits=splits)
        if causal:
            ref = prefix_attention(q.numpy(), kh, vh, kr, vr)
        else:
            ref = np.stack([decode_attention(q[:, i].numpy(), kh, vh, kr, vr)
                            for i in range(L)], axis=1)
        assert rel_err(out.cpu().numpy(), ref) <= 1e-3


@pytest.mark.parametrize("B,Hq,Hkv,D,G,Gv,R,T,L,splits,ring,half_q", [
    (2, 4, 1, 128, 32, 32, 64, 300, 5, 2, "bf16", True),     # 20 rows
    (1, 3, 1, 64, 64, 64, 64, 333, 30, 0, "f32", False),     # 90 rows
    (2, 2, 1, 256, 32, 32, 64, 200, 6, 0, "f16", False),     # 12 rows
    (1, 4, 2, 128, 32, 128, 64, 500, 70, 2, "f32", True),    # 280 rows
    (1, 3, 1, 128, 32, 32, 64, 20, 8, 0, "bf16", False),     # the window alone
])
def test_full_attention_and_masks_together(hip_device, B, Hq, Hkv, D, G, Gv, R, T, L, splits, ring,
                                           half_q):
    """causal=False (every row sees the whole context), and a first visible
    position together with holes, causal and not."""
    print(f"[rows] full: D={D} G={G} Gv={Gv} T={T} L={L} splits={splits} {ring}", flush=True)
    st, k, v = _store(hip_device, B, Hkv, D, G, Gv, R, T, L, ring)
    g = torch.Generator().manual_seed(L + D)
    q = torch.randn(B, Hq, L, D, generator=g)
    if half_q:
        q = q.bfloat16().float()
    total = st.quantized_tokens + st.res_len
    start = [min(41 * (b + 1), total - L) for b in range(B)]
    vis = torch.rand(B, total, generator=g) >= 0.2
    vis[:, total - L] = True
    kh, vh = oracle_history(k, v, st.n_chunks, G, Gv)
    q0 = st.n_chunks * G
    qn, kr, vr = q.transpose(1, 2).numpy(), k[:, :, q0:].numpy(), v[:, :, q0:].numpy()
    bound = _bound(qn, kh, kr)
    for mask, oracle in (({}, {}),
                         ({"kv_start": start, "key_mask": vis},
                          {"kv_start": np.array(start), "visible": vis.numpy()})):
        if mask:
            _check(st.attention(q.cuda(), num_splits=splits, **mask), q, st, k, v, G, Gv, **oracle)
        out = st.attention(q.cuda(), num_splits=splits, causal=False, **mask).cpu().numpy()
        for i in range(L):
            ref = decode_attention(qn[:, i], kh, vh, kr, vr, **oracle)
            size = decode_attention(qn[:, i], kh, np.abs(vh), kr, np.abs(vr), **oracle)
            assert (np.abs(out[:, i] - ref) <= bound * size).all()


def test_negative_scale_and_hidden_rows(hip_device):
    """A negative softmax scale turns the order of the scores; a sequence with
    every position hidden gives zeros."""
    st, k, v = _store(hip_device, 2, 1, 128, 32, 32, 64, 300, 8, "f32")
    q = torch.randn(2, 4, 8, 128, generator=torch.Generator().manual_seed(1))
    out = st.attention(q.cuda(), softmax_scale=-(128 ** -0.5))
    _check(out, -q, st, k, v, 32, 32)
    mask = torch.ones(2, st.quantized_tokens + st.res_len)
    mask[1] = 0
    out = st.attention(q.cuda(), key_mask=mask)
    assert torch.equal(out[1], torch.zeros_like(out[1])) and bool((out[0] != 0).any())


@pytest.mark.parametrize("ring,L", [("f32", 5), ("f32", 40), ("bf16", 5), ("bf16", 40)])
def test_infinite_window_elements(hip_device, ring, L):
    """An infinite key gives -inf scores (no weight) or poisons the rows that
    see it, an infinite value makes its channel infinite: what fp32 sums give,
    whatever the pieces."""
    Hq, D, R, T = 4, 128, 64, 200
    st, k, v = _store(hip_device, 1, 1, D, 32, 32, R, T, L, ring)
    q = torch.rand(1, Hq, L, D, generator=torch.Generator().manual_seed(2)) + 0.5
    q = q.bfloat16().float()
    t = st.res_len - L - 3                     # a window token every query sees
    slot = (st.res_start + t) % st.R
    st.k_res[0, 0, slot, 7] = -float("inf")    # scores -inf: the token drops out
    out = st.attention(q.cuda())
    total = st.quantized_tokens + st.res_len
    mask = torch.ones(1, total)
    mask[0, st.quantized_tokens + t] = 0
    kk = k.clone()
    _check(out, q, st, kk, v, 32, 32, visible=mask.numpy().astype(bool))
    st.k_res[0, 0, slot, 7] = 1.0
    st.v_res[0, 0, slot, 9] = float("inf")
    out = st.attention(q.cuda()).cpu()
    assert bool(torch.isinf(out[..., 9]).all())
    rest = torch.cat([out[..., :9], out[..., 10:]], -1)
    assert bool(torch.isfinite(rest).all())


ODD_CASES = [
    # Hq, D, G, Gv, T, L, splits, ring (B = Hkv = 1, R = 64)
    (4, 128, 32, 32, 40, 5, 0, "f32"),        # the window alone, 20 rows
    (4, 128, 32, 32, 40, 40, 0, "bf16"),      # the same, 160 rows
    (3, 64, 64, 64, 333, 7, 3, "f16"),        # G = 64, three splits
    (4, 64, 32, 64, 333, 30, 2, "f32"),       # 120 rows
    (4, 128, 64, 128, 600, 40, 2, "f32"),     # one value group
    (4, 256, 32, 256, 400, 3, 2, "f32"),      # head_dim 256, 12 rows
    (4, 256, 64, 128, 400, 30, 2, "bf16"),    # 120 rows
]


@pytest.mark.parametrize("Hq,D,G,Gv,T,L,splits,ring", ODD_CASES)
def test_infinite_key_comes_first(hip_device, Hq, D, G, Gv, T, L, splits, ring):
    """A token whose score is -inf takes no weight also where it is the first
    that a row sees: at the start of the context, after left padding, behind
    holes."""
    print(f"[rows] first -inf: D={D} G={G} Gv={Gv} T={T} L={L} {splits} {ring}", flush=True)
    st, k, v = _store(hip_device, 1, 1, D, G, Gv, 64, T, L, ring)
    q = torch.rand(1, Hq, L, D, generator=torch.Generator().manual_seed(2)) + 0.5
    q0 = st.quantized_tokens
    j = 3 if q0 else 0                          # the window token, and its position
    st.k_res[0, 0, (st.res_start + j) % st.R, 7] = -float("inf")
    pos, total = q0 + j, q0 + st.res_len
    vis = torch.ones(1, total, dtype=torch.bool)
    vis[0, pos] = False
    out = st.attention(q.cuda(), num_splits=splits)
    _check(out, q, st, k, v, G, Gv, visible=vis.numpy())
    out = st.attention(q.cuda(), num_splits=splits, kv_start=[pos])
    _check(out, q, st, k, v, G, Gv, kv_start=np.array([pos + 1]))
    holes = torch.arange(total)[None, :] >= pos
    out = st.attention(q.cuda(), num_splits=splits, key_mask=holes)
    _check(out, q, st, k, v, G, Gv, visible=(holes & vis).numpy())


@pytest.mark.parametrize("half_q", [False, True])
@pytest.mark.parametrize("Hq,D,G,Gv,T,L,splits,ring", ODD_CASES)
def test_window_elements_that_are_not_finite(hip_device, Hq, D, G, Gv, T, L, splits, ring, half_q):
    """An infinite or NaN window element touches what sees it and nothing else:
    not the rows it is hidden from (padding, or a token after theirs), nor, in a
    value, the other channels."""
    print(f"[rows] not finite: D={D} G={G} Gv={Gv} T={T} L={L} {splits} {ring} {half_q}", flush=True)
    st, k, v = _store(hip_device, 1, 1, D, G, Gv, 64, T, L, ring)
    q = torch.randn(1, Hq, L, D, generator=torch.Generator().manual_seed(L))
    if half_q:
        q = q.bfloat16().float()
    q0, n = st.quantized_tokens, st.res_len
    total = q0 + n
    vis = torch.ones(1, total, dtype=torch.bool)
    vis[0, q0 + 2] = False
    plain = st.attention(q.cuda(), num_splits=splits)
    inf, nan = float("inf"), float("nan")
    # two results of the bound's size apart, at most
    tol = 2 * _bound(q.transpose(1, 2).numpy(), k.numpy(), k.numpy()) * float(v.abs().max())

    def poisoned(t, key, value, **kw):
        slot = (st.res_start + t) % st.R
        saved = st.k_res[0, 0, slot].clone(), st.v_res[0, 0, slot].clone()
        if key is not None:
            st.k_res[0, 0, slot, 5] = key
        if value is not None:
            st.v_res[0, 0, slot, D - 3] = value
        out = st.attention(q.cuda(), num_splits=splits, **kw)
        st.k_res[0, 0, slot], st.v_res[0, 0, slot] = saved
        return out

    # hidden by holes, or before the first visible position
    for key, value in ((nan, nan), (inf, -inf), (-inf, inf)):
        _check(poisoned(2, key, value, key_mask=vis), q, st, k, v, G, Gv, visible=vis.numpy())
        _check(poisoned(2, key, value, kv_start=[q0 + 3]), q, st, k, v, G, Gv,
               kv_start=np.array([q0 + 3]))
    # the newest token: its own rows only
    out = poisoned(n - 1, nan, nan)
    assert bool(out[:, -1].isnan().all())
    assert float((out - plain)[:, :-1].abs().max()) <= tol
    # a value that every row sees: its channel only
    for value in (nan, inf):
        out = poisoned(0, None, value)
        assert not bool(out[..., D - 3].isfinite().any())
        out[..., D - 3] = plain[..., D - 3]
        assert float((out - plain).abs().max()) <= tol
    # a key: every row that sees it is NaN, or the token takes no weight
    out = poisoned(0, nan, None)
    assert bool(out.isnan().all())
    # finite keys whose scores overflow to -inf, first in sight
    if ring != "f16":
        qq = q.clone()
        qq[..., 5] = 1e3
        slot = st.res_start
        st.k_res[0, 0, slot, 5] = -3e38
        out = st.attention(qq.cuda(), num_splits=splits, kv_start=[q0])
        st.k_res[0, 0, slot, 5] = 0.0
        kk = k.clone()
        _check(out, qq, st, kk, v, G, Gv, kv_start=np.array([q0 + 1]))


@pytest.mark.parametrize("Hq,D,G,Gv,T,L,splits,ring", ODD_CASES[2:] + [
    (4, 128, 32, 32, 600, 5, 0, "f32"),       # 20 rows, four value groups
    (4, 256, 32, 32, 400, 30, 0, "f32"),      # eight value groups
])
def test_common_part_of_the_values(hip_device, Hq, D, G, Gv, T, L, splits, ring):
    """Values with a common offset of 20: packed values lose 3 * 2^-18 of their
    offset from the middle of their group's range (at most 1.5 scales), not of
    themselves.  Queries of one channel, so that a score is one product (6
    roundings of 2^-24, 2 more before the exponential): a weight is off by eps,
    which moves the output by eps * sum p |v - o|.  The output's fp32 sums round
    once per 32 tokens, and a few times at the end."""
    print(f"[rows] offset: D={D} G={G} Gv={Gv} T={T} L={L} {splits} {ring}", flush=True)
    st, k, v = _store(hip_device, 1, 1, D, G, Gv, 64, T, L, ring, v_offset=20.0)
    g = torch.Generator().manual_seed(L)
    q = torch.zeros(1, Hq, L, D)
    q[..., 11] = 3 * D ** 0.5 * torch.randn(1, Hq, L, generator=g)
    out = st.attention(q.cuda(), num_splits=splits).cpu().numpy().astype(np.float64)
    kh, vh = oracle_history(k, v, st.n_chunks, G, Gv)
    q0 = st.quantized_tokens
    qn, kr, vr = q.transpose(1, 2).numpy(), k[:, :, q0:].numpy(), v[:, :, q0:].numpy()
    ref = prefix_attention(qn, kh, vh, kr, vr)
    groups = v[:, :, :q0].reshape(1, 1, q0, D // Gv, Gv)
    scale = ((groups.amax(-1) - groups.amin(-1)) / 3).repeat_interleave(Gv, -1).numpy()
    part = 1.5 * prefix_attention(qn, kh, scale, kr, 0 * vr)
    square = prefix_attention(qn, kh, vh.astype(np.float64) ** 2, kr, vr.astype(np.float64) ** 2)
    spread = np.sqrt(np.maximum(square - ref ** 2, 0))          # >= sum p |v - o|
    smax = float(np.abs(qn).max() * np.abs(k.numpy()).max()) * D ** -0.5
    eps = 2 * (8 * 2.0 ** -24 * smax + 2.0 ** -22)
    units = (T + L) / 32 + 8
    bound = 3 * 2.0 ** -18 * part + eps * spread + units * 2.0 ** -24 * np.abs(ref)
    err = np.abs(out - ref) / bound
    print(f"[rows]   largest error {err.max():.2f} of the bound", flush=True)
    assert err.max() <= 1


@pytest.mark.parametrize("Hq,D,G,Gv,T,L,splits,ring", ODD_CASES)
def test_a_query_that_is_not_finite_stays_in_its_row(hip_device, Hq, D, G, Gv, T, L, splits, ring):
    st, k, v = _store(hip_device, 1, 1, D, G, Gv, 64, T, L, ring)
    q = torch.randn(1, Hq, L, D, generator=torch.Generator().manual_seed(L))
    plain = st.attention(q.cuda(), num_splits=splits)
    tol = 2 * _bound(q.transpose(1, 2).numpy(), k.numpy(), k.numpy()) * float(v.abs().max())
    for x in (float("nan"), float("inf")):
        bad = q.clone()
        bad[0, 1, L // 2, 3] = x
        out = st.attention(bad.cuda(), num_splits=splits)
        assert bool(out[0, L // 2, 1].isnan().all())
        out[0, L // 2, 1] = plain[0, L // 2, 1]
        assert float((out - plain).abs().max()) <= tol
