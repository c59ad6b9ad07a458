"""GPU parity of the plain-layout attention kernel (stores whose geometry the
matrix-core code order does not cover) at the edges of its lane mapping: 4, 2 or
1 lanes per token (G 16, 32, 48 and 64), code words that do not divide among
them (head_dim 80, 240), idle lanes (G 48, small head dims), value groups
smaller and larger than the key group, 1 to 8 query rows with padding, window
passes with idle lanes, splits, several query tokens and hidden positions.

Everything is fp32, so the bound is that of fp32 sums whose roundings (2^-25 of
the running sum, rms) are independent, at six standard deviations.  A score is a
sum of 2 D terms q ks c and q kz, none of its running sums larger than S = scale *
sum_d |q_d| max_t |k_d|: off by sqrt(2 D) 2^-25 S, which moves a weight and the
normaliser by as much.  The output is a sum over the T tokens of terms up to 3
max|v| (p vs c and p vz before they cancel): off by sqrt(T) 2^-25 * 3 max|v|.
"""

import numpy as np
import pytest
import torch

from oracle.attention import decode_attention, prefix_attention
from tests.kv_helpers import make_kv, oracle_history

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, D, G, Gv, R, T, splits, ring
    (1, 1, 1, 16, 16, 16, 32, 150, 0, "f32"),        # one code word per token
    (2, 6, 2, 80, 16, 16, 32, 500, 3, "bf16"),       # 5 words over 4 lanes, 3 rows of 4
    (1, 8, 1, 96, 32, 32, 64, 700, 0, "f32"),        # 8 rows
    (2, 4, 4, 48, 48, 16, 96, 400, 2, "f16"),        # G 48: one lane per token, 16 idle
    (1, 4, 2, 112, 32, 112, 64, 300, 0, "f32"),      # one value group per token
    (1, 8, 2, 128, 16, 8, 64, 333, 4, "bf16"),       # small value groups, 4 rows
    (1, 2, 1, 80, 64, 16, 128, 600, 0, "f32"),       # G 64
    (1, 3, 1, 240, 48, 80, 96, 500, 2, "f32"),       # head_dim 240: 15 words, 3 dwords a channel
    (2, 12, 1, 64, 16, 16, 32, 20, 0, "bf16"),       # no chunk yet, two head groups
    (1, 2, 2, 256, 16, 64, 64, 400, 0, "f32"),       # head_dim 256
    (1, 2, 2, 128, 32, 8, 64, 300, 0, "f32"),        # 512 value factors: the generic kernel
    (4, 8, 1, 80, 64, 80, 128, 2000, 0, "bf16"),     # 8 rows of 64 tokens: the generic kernel
    (4, 32, 8, 48, 48, 16, 96, 2000, 0, "f32"),      # 4 rows of 144 factors: likewise
    (4, 32, 8, 96, 64, 96, 128, 1000, 0, "f16"),     # 4 rows, a workgroup for every CU
]


def _bound(q, kh, vh, kr, vr):
    keys, vals = np.concatenate([kh, kr], 2), np.concatenate([vh, vr], 2)
    D, T = keys.shape[3], keys.shape[2]
    kmax, vmax = np.abs(keys).max(2), np.abs(vals).max()
    qa = np.abs(q).reshape(q.shape[0], -1, q.shape[-2] if q.ndim == 3 else q.shape[2], D)
    g = qa.shape[2] // kmax.shape[1]
    s = max(float((qa[b, :, h] @ kmax[b, h // g]).max())
            for b in range(qa.shape[0]) for h in range(qa.shape[2]))
    return 6 * 2.0 ** -25 * (2 * (2 * D) ** 0.5 * s * D ** -0.5 + 3 * T ** 0.5) * vmax


@pytest.mark.parametrize("B,Hq,Hkv,D,G,Gv,R,T,splits,ring", CASES)
def test_plain_kernel_matches_oracle(hip_device, B, Hq, Hkv, D, G, Gv, R, T, splits, ring):
    from intel_kivi_hybrid_amd.store import PackedKVStore
    print(f"[plain] B={B} Hq={Hq} Hkv={Hkv} D={D} G={G} Gv={Gv} R={R} T={T} splits={splits} {ring}",
          flush=True)
    dt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[ring]
    k, v = (x.to(dt).float() for x in make_kv(B, Hkv, T, D, seed=T + D))
    st = PackedKVStore(B, Hkv, D, G, R, "cuda:0", group_size_v=Gv, residual_dtype=dt)
    assert st.code_layout == 0
    st.extend(k.to("cuda", dt), v.to("cuda", dt), flush_at=R)
    g = torch.Generator().manual_seed(D + T)
    q = torch.randn(B, Hq, D, generator=g)
    kh, vh = oracle_history(k, v, st.n_chunks, G, Gv)
    q0 = st.n_chunks * G
    kr, vr = k[:, :, q0:].numpy(), v[:, :, q0:].numpy()

    def check(out, ref, bound):
        err = float(np.abs(out.cpu().numpy().astype(np.float64) - ref).max())
        print(f"[plain]   largest error {err:.2e} (bound {bound:.2e})", flush=True)
        assert err <= bound

    bound = _bound(q.numpy(), kh, vh, kr, vr)
    out = st.attention(q.cuda(), num_splits=splits)
    check(out, decode_attention(q.numpy(), kh, vh, kr, vr), bound)
    assert torch.equal(out, st.attention(q.cuda(), num_splits=splits))
    vis = torch.rand(B, T, generator=g) >= 0.3
    vis[:, -1] = True
    check(st.attention(q.cuda(), num_splits=splits, key_mask=vis),
          decode_attention(q.numpy(), kh, vh, kr, vr, visible=vis.numpy()), bound)
    start = [min(29 * (b + 1), T - 4) for b in range(B)]
    check(st.attention(q.cuda(), num_splits=splits, kv_start=start),
          decode_attention(q.numpy(), kh, vh, kr, vr, kv_start=np.array(start)), bound)
    L = 3
    ql = torch.randn(B, Hq, L, D, generator=g)
    qn = ql.transpose(1, 2).numpy()
    check(st.attention(ql.cuda(), num_splits=splits), prefix_attention(qn, kh, vh, kr, vr),
          _bound(qn, kh, vh, kr, vr))
