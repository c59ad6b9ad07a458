"""GPU check of the plain-layout flush kernel at the edges of its rule: 1 to 8
tokens per thread, segments that do not divide the chunk, value groups of 1 to
64 lanes, rows as wide as the workgroup, and (last two shapes) a value group
that is no power of two of lanes and too many tokens per thread, which the
general kernel takes.

Bar: bit-exact codes, scales, zeros and history against the oracle's."""

import pytest
import torch

from tests.kv_helpers import check_store_bit_exact, make_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,G,Gv", [
    (8, 4, 4), (20, 12, 4), (48, 20, 16), (80, 16, 16), (96, 32, 32), (64, 16, 16), (72, 16, 8),
    (96, 64, 32), (256, 12, 256), (1024, 8, 64), (320, 16, 64), (96, 32, 96), (520, 12, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_plain_flush_is_bit_exact(hip_device, D, G, Gv, dtype):
    from intel_kivi_hybrid_amd.store import PackedKVStore
    print(f"[flush] D={D} G={G} Gv={Gv} {dtype}", flush=True)
    B, H, R = 2, 2, G + 3
    T = 5 * G + 7
    k, v = make_kv(B, H, T, D, seed=D + G)
    for x in (k, v):
        x[0, 0, 1] = 0.0                          # constant value groups, signed zeros
        x[0, 0, 1, ::2] = -0.0
        x[0, 1, :, 3] = 0.5                       # a constant key group
        x[1, 0, 2, 1] = float("nan")              # code 0
        if dtype == torch.float32:
            x[1, 1, 4, 0] = 3e36                  # past the reference's initial minimum
    k, v = k.to(dtype), v.to(dtype)
    st = PackedKVStore(B, H, D, G, R, "cuda:0", group_size_v=Gv, keep_history=True)
    st.extend(k[:, :, :G + 1].cuda(), v[:, :, :G + 1].cuda(), flush_at=R)   # all in the ring
    st.extend(k[:, :, G + 1:].cuda(), v[:, :, G + 1:].cuda(), flush_at=R)   # ring, both, new
    assert st.n_chunks == (T - R) // G + 1
    check_store_bit_exact(st, k.float(), v.float())
