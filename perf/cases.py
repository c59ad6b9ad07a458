"""The work that users of this package have it do, as timed cases.

Five kinds of call, each through the package's public entry points:

* ``decode``: one decode step of one attention layer on a ``PackedKVStore``
  (the step's token staged, fused attention over [packed history ; window],
  the token dropped again so that a pass leaves the store as it found it).
* ``layer``: one forward of ``new`` tokens of one attention layer through a
  ``KiviPackedCache``, as a transformers model makes it (``update()``, the
  registered attention function, ``crop()``): one token is a decode step, a
  few a verification pass of drafted tokens, hundreds a chunk of a long prompt.
* ``prompt``: a prompt's K/V quantised into an empty store.
* ``codec``: the reference's ops on whole K and V tensors (quantise, then
  dequantise).
* ``served``: a session of a ``KiviCache`` served to a model's own attention.

K/V are N(0,1) with four outlier channels per kv head in the keys and 2 % of
outlier tokens in the values; queries are N(0,1), so natural-unit scores have
a standard deviation of about 2.
"""

import math

import torch

from intel_kivi_hybrid_amd import KiviCache, _C
from intel_kivi_hybrid_amd.cache.packed_cache import (KiviPackedCache,
                                                      kivi_packed_attention_forward)
from intel_kivi_hybrid_amd.store import PackedKVStore

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _attn(name, kind, B, Hq, Hkv, D, T, R=128, G=32, Gv=None, dtype="f32", new=1, pad="none"):
    """An attention case: T tokens of context already held when the call's
    ``new`` tokens arrive."""
    case = {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "D": D, "T": T, "R": R, "G": G,
            "Gv": G if Gv is None else Gv, "dtype": dtype, "new": new, "pad": pad}
    return {"name": name, **case} if name else case


def _prompt(name, B, H, D, T, R=128, G=32, Gv=None, dtype="bf16"):
    case = {"kind": "prompt", "B": B, "H": H, "D": D, "T": T, "R": R, "G": G,
            "Gv": G if Gv is None else Gv, "dtype": dtype}
    return {"name": name, **case} if name else case


def _codec(name, B, H, T, D, G):
    case = {"kind": "codec", "B": B, "H": H, "T": T, "D": D, "G": G}
    return {"name": name, **case} if name else case


def _served(name, layers, B, H, D, T, steps, R, G):
    case = {"kind": "served", "layers": layers, "B": B, "H": H, "D": D, "T": T, "steps": steps,
            "R": R, "G": G}
    return {"name": name, **case} if name else case


def listed():
    return [
        # One layer of a GPT-2-sized model generating for one user: the
        # smallest call, all latency and host time.
        _attn("layer_step_small", "layer", 1, 12, 12, 64, 300, R=64),
        # One user's long chat on a Llama-3-8B-shaped model (bf16 K/V).
        _attn("decode_single", "decode", 1, 32, 8, 128, 8150, dtype="bf16"),
        # The benchmark's serving batch: 64 sequences at 8K context, fp32 window.
        _attn("decode_serving", "decode", 64, 32, 8, 128, 8191),
        # A mid-sized batch of a 70B-shaped model, 8 query heads per kv head.
        _attn("decode_gqa8", "decode", 16, 64, 8, 128, 7777, dtype="bf16"),
        # A left-padded batch of unequal prompts on a multi-head (7B-shaped) model.
        _attn("decode_padded_mha", "decode", 16, 32, 32, 128, 4187, pad="left"),
        # A few documents at 128K context, one value group per token.
        _attn("decode_long", "decode", 4, 32, 8, 128, 131071 + 96, Gv=128),
        # A multi-head model whose head_dim is not a power of two (its store
        # keeps the plain code order).
        _attn("decode_head96", "decode", 4, 32, 32, 96, 4000),
        # The verification pass of assisted decoding: 4 drafted tokens and one more.
        _attn("layer_verify", "layer", 8, 32, 8, 128, 4097, dtype="bf16", new=5),
        # A chunk of a long prompt fed to a cache that already holds 8K tokens.
        _attn("layer_chunk", "layer", 1, 32, 8, 128, 8100, dtype="bf16", new=512),
        # A batch of prompts entering the cache after their prefill.
        _prompt("prompt_flush", 16, 8, 128, 4111),
        # The reference's ops over a whole batch's K and V (8 x 32 heads x 4096 x 128).
        _codec("codec_full", 8, 32, 4096, 128, 32),
        # The reference's own flow: 12 layers, a short prompt, 40 tokens served
        # to the model's attention (one flush on the way).
        _served("served_session", 12, 1, 12, 64, 40, 40, 64, 32),
    ]


# Head layouts (query heads, kv heads) of the models the tests and the
# benchmark are shaped after.
_HEADS = [(32, 8), (32, 32), (12, 12), (64, 8), (24, 8), (16, 2), (28, 4), (16, 4)]
# (head_dim, G, Gv): the matrix-core code order, then the plain one.
_GEOMETRIES = [(128, 32, 32), (128, 32, 32), (128, 32, 128), (128, 64, 64), (64, 32, 32),
               (64, 64, 64), (256, 32, 32), (96, 32, 32), (80, 16, 16), (64, 16, 16)]

_MOST_STORE_ELEMS = 64 * 8 * 8192 * 128           # per tensor: the serving batch
_MOST_CHUNK_SCORES = 512 * 32 * 8700 * 128        # q_len x heads x context x head_dim


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "layer", "layer", "prompt", "codec",
                       "served"])
    if kind == "codec":
        D, G = rng.choice([(128, 32), (64, 32), (128, 64), (96, 32), (64, 16), (128, 128)])
        B, H = _log_int(rng, 1, 8), rng.choice([8, 12, 32])
        T = G * _log_int(rng, 1, 4096 // G)
        return _codec(None, B, H, T, D, G)
    if kind == "served":
        D, G = rng.choice([(64, 32), (128, 32), (64, 64)])
        return _served(None, rng.choice([2, 6, 12]), rng.choice([1, 1, 2]), rng.choice([8, 12]),
                       D, _log_int(rng, 7, 300), rng.randint(5, 40), rng.choice([64, 128]), G)
    D, G, Gv = rng.choice(_GEOMETRIES)
    R = rng.choice([64, 128])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "prompt":
        B, H = _log_int(rng, 1, 16), rng.choice([8, 12])
        return _prompt(None, B, H, D, _log_int(rng, 33, 4200), R, G, Gv, dtype)
    Hq, Hkv = rng.choice(_HEADS)
    B = _log_int(rng, 1, 64 if kind == "decode" else 8)
    most = max(256, min(131072 if kind == "decode" else 16384,
                        _MOST_STORE_ELEMS // (B * Hkv * D)))
    T = _log_int(rng, 40, most)
    new, pad = 1, "none"
    if kind == "layer":
        most_new = min(512, _MOST_CHUNK_SCORES // (B * Hq * D * (T + 512)))
        new = rng.choice([1, 2, _log_int(rng, 2, max(2, most_new)),
                          _log_int(rng, 2, max(2, most_new))])
    else:
        pad = rng.choice(["none", "none", "none", "left", "holes"])
    if kind == "layer" and new == 1 and T >= R and (T - R) % G == G - 1:
        T += 1                # (a window the step does not fill: see run())
    elif kind == "layer" and new == 1 and T == R - 1:
        T -= 1
    return _attn(None, kind, B, Hq, Hkv, D, T, R, G, Gv, dtype, new, pad)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed, part):
    return torch.Generator(device=DEVICE).manual_seed(1_000_003 * seed + part)


def _kv(B, H, T, D, seed, part=0):
    """K and V ``[B, H, T, D]`` fp32 on the GPU, with outliers."""
    g = _generator(seed, part)
    k = torch.randn(B, H, T, D, generator=g, device=DEVICE)
    v = torch.randn(B, H, T, D, generator=g, device=DEVICE)
    ch = torch.rand(H, D, generator=g, device=DEVICE).topk(min(4, D), dim=-1).indices
    k *= torch.ones(H, D, device=DEVICE).scatter_(1, ch, 10.0)[None, :, None, :]
    v *= 1.0 + 7.0 * (torch.rand(B, H, T, 1, generator=g, device=DEVICE) < 0.02)
    return k, v


def _attn_inputs(case, seed):
    """Context K/V, the call's new K/V and queries, in the model's type."""
    dt = DTYPES[case["dtype"]]
    k, v = _kv(case["B"], case["Hkv"], case["T"] + case["new"], case["D"], seed)
    k, v = k.to(dt), v.to(dt)
    q = torch.randn(case["B"], case["Hq"], case["new"], case["D"],
                    generator=_generator(seed, 1), device=DEVICE)
    if case["kind"] == "layer":
        q = q.to(dt)
    return k, v, q


def _hidden_mask(case, seed):
    """Visible positions ``[B, T + 1]`` of a padded batch (None: all)."""
    B, T = case["B"], case["T"] + 1
    g = torch.Generator().manual_seed(seed + 77)
    if case["pad"] == "left":
        start = torch.randint(0, max(1, T // 2), (B,), generator=g)
        start[0] = 0
        return torch.arange(T)[None, :] >= start[:, None]
    if case["pad"] == "holes":
        vis = torch.rand(B, T, generator=g) >= 0.1
        vis[:, -1] = True
        return vis
    return None


def prepare(case, seed):
    kind = case["kind"]
    if kind == "codec":
        B, H, T, D, G = (case[n] for n in ("B", "H", "T", "D", "G"))
        k, v = _kv(B, H, T, D, seed)
        n = k.numel()
        gv = min(G, D)
        out = {"case": case, "k": k.transpose(2, 3).contiguous(), "v": v, "gv": gv}
        for x, g in (("k", G), ("v", gv)):
            out[x + "_codes"] = torch.empty(n // 4, dtype=torch.uint8, device=DEVICE)
            out[x + "_scale"] = torch.empty(n // g, device=DEVICE)
            out[x + "_zero"] = torch.empty(n // g, device=DEVICE)
            out[x + "_hat"] = torch.empty(n, device=DEVICE)
        return out
    if kind == "prompt":
        B, H, D, T = (case[n] for n in ("B", "H", "D", "T"))
        dt = DTYPES[case["dtype"]]
        # (a model's projections are token-major: K/V arrive as transposed views)
        k, v = (x.to(dt).transpose(1, 2).contiguous().transpose(1, 2)
                for x in _kv(B, H, T, D, seed))
        st = PackedKVStore(B, H, D, case["G"], case["R"], DEVICE, group_size_v=case["Gv"],
                           chunk_capacity=T // case["G"] + 1, residual_dtype=dt)
        return {"case": case, "store": st, "k": k, "v": v}
    if kind == "served":
        L, B, H, D, T, S = (case[n] for n in ("layers", "B", "H", "D", "T", "steps"))
        kvs = [_kv(B, H, T + S, D, seed, part=10 + i) for i in range(L)]
        cache = KiviCache(L, D, H, device=DEVICE, group_size=case["G"],
                          residual_length=case["R"])
        return {"case": case, "cache": cache,
                "prompt": tuple((k[:, :, :T].contiguous(), v[:, :, :T].contiguous())
                                for k, v in kvs),
                "steps": [[(k[:, :, T + s:T + s + 1].contiguous(),
                            v[:, :, T + s:T + s + 1].contiguous()) for k, v in kvs]
                          for s in range(S)]}
    k, v, q = _attn_inputs(case, seed)
    T, G, R, D = case["T"], case["G"], case["R"], case["D"]
    kn, vn = k[:, :, T:].contiguous(), v[:, :, T:].contiguous()
    state = {"case": case, "k": kn, "v": vn, "q": q}
    if kind == "layer":
        cache = KiviPackedCache(1, D, case["Hkv"], device=DEVICE, group_size=G,
                                residual_length=R, value_group_size=case["Gv"],
                                chunk_capacity=T // G + 1)
        cache.update(k[:, :, :T], v[:, :, :T], 0)
        state["cache"] = cache
        return state
    st = PackedKVStore(case["B"], case["Hkv"], D, G, R, DEVICE, group_size_v=case["Gv"],
                       chunk_capacity=T // G + 1, residual_dtype=DTYPES[case["dtype"]])
    st.extend(k[:, :, :T], v[:, :, :T], flush_at=R)
    state["store"], state["q"] = st, q[:, :, 0].contiguous()
    vis = _hidden_mask(case, seed)
    if case["pad"] == "left":
        state["kv_start"] = vis.int().argmax(-1).to(torch.int32).to(DEVICE)
    elif case["pad"] == "holes":
        # (the mask's words are made once per forward, for every layer)
        state["hidden"] = _C.hidden_positions(vis, DEVICE)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        st = state["store"]
        st.stage_token(state["k"], state["v"])
        o = st.attention(state["q"], kv_start=state.get("kv_start"), hidden=state.get("hidden"))
        st.rollback(1)
        return o
    if kind == "layer":
        cache = state["cache"]
        k, v = cache.update(state["k"], state["v"], 0)
        o, _ = kivi_packed_attention_forward(None, state["q"], k, v, None,
                                             scaling=case["D"] ** -0.5)
        cache.layers[0].crop(-case["new"])
        return o
    if kind == "prompt":
        st = state["store"]
        st.reset()
        st.extend(state["k"], state["v"], flush_at=case["R"])
        n = st.n_chunks
        kr, vr = st.residual()
        return [st.k_codes[:, :, :n], st.k_scale[:, :, :n], st.k_zero[:, :, :n],
                st.v_codes[:, :, :n], st.v_scale[:, :, :n], st.v_zero[:, :, :n], kr, vr]
    if kind == "codec":
        s, G, gv, D = state, case["G"], state["gv"], case["D"]
        _C.quantize_keys_async(s["k"], s["k_codes"], s["k_scale"], s["k_zero"], G)
        _C.quantize_values_async(s["v"], s["v_codes"], s["v_scale"], s["v_zero"], D, gv)
        _C.dequantize_keys_async(s["k_codes"], s["k_scale"], s["k_zero"], s["k_hat"], G)
        _C.dequantize_values_async(s["v_codes"], s["v_scale"], s["v_zero"], s["v_hat"], D, gv)
        return [s[n] for n in ("k_codes", "k_scale", "k_zero", "k_hat",
                               "v_codes", "v_scale", "v_zero", "v_hat")]
    cache = state["cache"]
    cache.reset()
    cache.add_tokens(state["prompt"])
    for step in state["steps"]:
        past = cache.get_full_cache()
        for i, (k, v) in enumerate(step):
            past.update(k, v, i)               # what the model's attention does
        cache.add_tokens(past)
    return [t for layer in cache.get_full_cache().layers for t in (layer.keys, layer.values)]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _chunks(T, R, G):
    """Chunks quantised once T tokens have passed through a window of R."""
    return 0 if T < R else (T - R) // G + 1


def work(case):
    kind = case["kind"]
    if kind == "codec":
        n = case["B"] * case["H"] * case["T"] * case["D"]
        gv = min(case["G"], case["D"])
        code = [n // 4 + 8 * n // g for g in (case["G"], gv)]
        return {"bytes": 2 * (4 * n + 4 * n) + 2 * sum(code), "flops": 2 * 10 * n}
    if kind == "prompt":
        B, H, D, T, G = (case[x] for x in ("B", "H", "D", "T", "G"))
        e = DTYPES[case["dtype"]].itemsize
        q = _chunks(T, case["R"], G) * G
        per = 2 * T * D * e + 2 * q * D // 4 + 8 * q * D // G + 8 * q * D // case["Gv"] \
            + 2 * (T - q) * D * e
        return {"bytes": B * H * per, "flops": 2 * 10 * B * H * q * D}
    if kind == "served":
        L, B, H, D, T, S = (case[x] for x in ("layers", "B", "H", "D", "T", "steps"))
        # each step: the new token in, and the served K/V of the whole context
        # handed to the model once (written once when a flush changes it)
        total = T + S
        flushes = _chunks(total, case["R"], case["G"])
        per = 2 * 4 * D * (total + (1 + flushes) * total)
        return {"bytes": L * B * H * per, "flops": L * B * H * 2 * 10 * flushes * case["G"] * D}
    B, Hq, Hkv, D, T, n = (case[x] for x in ("B", "Hq", "Hkv", "D", "T", "new"))
    G, Gv, e = case["G"], case["Gv"], DTYPES[case["dtype"]].itemsize
    q = _chunks(T, case["R"], G) * G
    res = T - q + n
    per = 2 * q * D // 4 + 8 * q * D // G + 8 * q * D // Gv + 2 * e * res * D + 2 * e * n * D
    io = 2 * B * Hq * n * D * (e if kind == "layer" else 4)
    return {"bytes": B * Hkv * per + io, "flops": 4 * B * Hq * n * (T + n / 2) * D}


def tolerance(case):
    if case["kind"] in ("codec", "prompt", "served"):
        return "exact"           # codes, scales, zeros and served values are fixed bits
    if case["kind"] == "layer" and case["dtype"] == "bf16":
        return {"rel": 7e-3}     # the output itself is rounded to bf16: 1.7e-3 measured
    return {"rel": 2e-4}         # 1e-5 to 6e-5 measured, the most at 128K context


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _quantise(x, dim):
    """(codes, scale, zero) of groups along ``dim``: the 2-bit format's own
    fp32 rule, which decides the codes."""
    three = torch.full((1,), 3.0, device=x.device)
    lo, hi = x.amin(dim, keepdim=True), x.amax(dim, keepdim=True)
    scale = (hi - lo) / three + 1e-10
    t = (x - lo) / scale
    down = t.floor()                  # (t + 0.5 would round the float below 0.5 up)
    return (down + ((t - down) >= 0.5)).clamp(0, 3), scale, lo


def _history(k, v, n, G, Gv):
    """float64 K/V of n tokens as the packed store holds them, ``[.., n, D]``."""
    shape, D = k.shape, k.shape[-1]
    c, s, z = _quantise(k.float().reshape(*shape[:-2], n // G, G, D), -2)
    k_hat = (c.double() * s.double() + z.double()).reshape(shape)
    c, s, z = _quantise(v.float().reshape(*shape[:-1], D // Gv, Gv), -1)
    return k_hat, (c.double() * s.double() + z.double()).reshape(shape)


def _exact_attention(case, seed):
    B, Hq, Hkv, D, T, n = (case[x] for x in ("B", "Hq", "Hkv", "D", "T", "new"))
    G, Gv = case["G"], case["Gv"]
    k, v, q = _attn_inputs(case, seed)
    nq = _chunks(T, case["R"], G) * G
    vis = _hidden_mask(case, seed)
    out = torch.empty(B, n, Hq, D, dtype=torch.float64, device=DEVICE)
    pos = torch.arange(T + n, device=DEVICE)
    causal = pos[None, :] <= T + torch.arange(n, device=DEVICE)[:, None]
    for b in range(B):
        for h in range(Hkv):
            kh, vh = k[b, h, nq:].double(), v[b, h, nq:].double()
            if nq:
                ka, va = _history(k[b, h, :nq], v[b, h, :nq], nq, G, Gv)
                kh, vh = torch.cat([ka, kh]), torch.cat([va, vh])
            heads = slice(h * (Hq // Hkv), (h + 1) * (Hq // Hkv))
            s = q[b, heads].double() @ kh.T.contiguous() * D ** -0.5       # [heads, n, T + n]
            keep = causal if vis is None else causal & vis[b].to(DEVICE)[None, :]
            s = s.masked_fill(~keep, -math.inf)
            out[b, :, heads] = (s.softmax(-1) @ vh).transpose(0, 1)
    return out[:, 0] if case["kind"] == "decode" else out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "layer"):
        return _exact_attention(case, seed)
    if kind == "codec":
        B, H, T, D, G = (case[x] for x in ("B", "H", "T", "D", "G"))
        k, v = _kv(B, H, T, D, seed)
        out = []
        for x in (k.transpose(2, 3).reshape(-1, G), v.reshape(-1, min(G, D))):
            c, _, _ = _quantise(x, -1)
            lo, hi = x.double().amin(-1, keepdim=True), x.double().amax(-1, keepdim=True)
            s = (hi - lo) / 3 + 1e-10
            out += [None, s.reshape(-1), lo.reshape(-1), (c.double() * s + lo).reshape(-1)]
        return out
    if kind == "prompt":
        B, H, D, T, G, Gv = (case[x] for x in ("B", "H", "D", "T", "G", "Gv"))
        k, v = (x.to(DTYPES[case["dtype"]]).double() for x in _kv(B, H, T, D, seed))
        n = _chunks(T, case["R"], G)
        q = n * G
        kc = k[:, :, :q].reshape(B, H, n, G, D)
        vc = v[:, :, :q].reshape(B, H, n, G, D // Gv, Gv)
        klo, khi, vlo, vhi = kc.amin(3), kc.amax(3), vc.amin(-1), vc.amax(-1)
        return [None, (khi - klo) / 3 + 1e-10, klo,
                None, ((vhi - vlo) / 3 + 1e-10).transpose(-1, -2), vlo.transpose(-1, -2),
                k[:, :, q:], v[:, :, q:]]
    L, B, H, D, T, S = (case[x] for x in ("layers", "B", "H", "D", "T", "steps"))
    out = []
    for i in range(L):
        k, v = _kv(B, H, T + S, D, seed, part=10 + i)
        nq = _chunks(T + S, case["R"], case["G"]) * case["G"]
        ka, va = _history(k[:, :, :nq], v[:, :, :nq], nq, case["G"], case["G"])
        out += [torch.cat([ka, k[:, :, nq:].double()], 2),
                torch.cat([va, v[:, :, nq:].double()], 2)]
    return out
