// Packed-KV attention for many query rows per kv head (gfx950 matrix cores).
//
// Causal or full attention of q_len query tokens per sequence over [packed
// chunks ; residual window] (kivi_packed_attention) when q_len * (q_heads /
// kv_heads) exceeds the 8 rows that one launch of the decode kernel
// (kivi_attention_mfma.hpp) takes: the verification pass of drafted tokens, a
// chunk of a long prompt.  The decode kernel multiplies the codes themselves,
// which needs the query folded with each chunk's key scales, work per row and
// chunk; with many rows the other order is cheaper: dequantise each 32 tokens
// once and let every row use them.
//
// * Row r of a kv head is query token r / hg, head r % hg.  Rows are held in
//   tiles of 16, and the context is walked in units of 32 tokens: the packed
//   chunks' (a G = 64 chunk is two units), then the window's.
// * K_hat and V_hat are expanded into MFMA A operands as bf16 pieces (hi + mid
//   + lo for keys and for the fp32 window's values, hi + lo for packed
//   values): a packed code word already holds one lane's codes of two tiles.
//   Packed values enter as their offset (c - 1.5) vs from the middle of their
//   group's range; the middles vz + 1.5 vs, one per token and group, are rows of
//   a tile of their own, whose sums are added at the end (Rows::middles).
// * Scores are formed transposed, S^T = K_hat Q^T, so a lane holds the scores
//   of one query row (its l % 16) for 8 of the unit's tokens, and the output
//   transposed too, O^T = V_hat^T P^T: a row's softmax state and rescale are
//   per-lane scalars, and the probabilities go from the score registers into
//   the second product's B operand without moving between lanes.
// * Precision: products of pieces are accumulated in fp32.  A query whose
//   values are all bf16 (a bf16 model's, widened) takes one piece and three
//   products per key tile, any other query three pieces and six products
//   (~2^-24 relative); packed values' offsets take three products of two
//   pieces (~2^-17 of p vs per token, averaged over the context), their
//   groups' middles and window values six of three: a common part of the
//   values, which does not average out, keeps fp32's precision (32/8 heads, 2K
//   tokens, fp32, error relative to float64: zero-mean values 4.2e-6, with an
//   offset of 20 sigma 1.7e-7; the decode launches 7.5e-6 and 4.9e-7).  The softmax
//   is online in fp32, in the log2 domain; its maximum moves only when exceeded by
//   more than 8 (weights <= 256).
// * Elements that are not finite as bf16 have no pieces (inf - inf): every sum
//   that they enter comes out NaN.  A workgroup whose window sums come out NaN
//   walks its range again with the window in plain fp32 (Rows::plain_unit):
//   an infinite value makes its channel infinite, a score of -inf gives its
//   token no weight, and a token that a row does not see does not touch it.
//   Packed chunks keep the same walk: non-finite factors make the rows that
//   see them NaN.
//
// Two kernels (few_rows(): which rows take which):
// * attn_rows_shared_kernel (many rows): eight waves with up to 32 rows each
//   expand every unit together into LDS and read it from there.
// * attn_rows_wave_kernel (few rows): each wave takes units of its own and
//   expands them straight into its operand registers.
//
// Measured (MI355X, 32/8 heads, head_dim 128, us per call; the decode kernel's
// launches before, this file's after): 512 query tokens over 8.1K packed tokens,
// B=1: 256 launches, 4810 -> 233, fp32 queries 4740 -> 340; 5 tokens over 4K, B=8: 3
// launches, 78 -> 45, fp32 77 -> 49.
#include <float.h>
#include <math.h>

#include "kivi_attention.hpp"
#include "kivi_common.hpp"
#include "kivi_mfma.hpp"

namespace kivi {
namespace {

constexpr int kUnit = 32;                   // tokens per step
constexpr float kMoveMax = 8.0f;            // log2 units
constexpr int kWindowWeight = 2;            // cost of a window unit in packed units
constexpr int kKP = 3;                      // key pieces
constexpr int kVPWin = 3, kVPChunk = 2;     // value pieces: window, packed chunks
constexpr int kPP = 3;                      // weight pieces
constexpr int kTile = kWave * 16;           // bytes of one operand tile

template <bool V>
struct BoolC {
    static constexpr bool value = V;
};

// max / sum over the four lanes that share a query row (l % 16)
__device__ __forceinline__ float row4_max(float v) {
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float row4_sum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

__device__ __forceinline__ int64_t out_offset(const RowsLaunch& a, int b, int kvh, int r) {
    return (((int64_t)b * a.q_len + r / a.hg) * a.Hq + (int64_t)kvh * a.hg + r % a.hg) * a.D;
}
__device__ __forceinline__ int64_t query_offset(const RowsLaunch& a, int b, int kvh, int r) {
    return b * a.q_sb + r / a.hg * a.q_st + ((int64_t)kvh * a.hg + r % a.hg) * a.q_sh;
}

// Queries and outputs are in the caller's type, read and written here: a bf16
// model's step otherwise pays up to three more launches (q widened, q made
// token-major, the output rounded), 7 us of 51 for 5 query tokens over 4K, B=8,
// 10 of 228 for 512 tokens over 8.1K, B=1 (32/8 heads, head_dim 128).
// f(load) with load(i): elements i .. i + 3 of the queries, widened exactly.
// (one branch around all loads: a branch per load would wait for each)
template <class F>
__device__ __forceinline__ void with_query(const RowsLaunch& a, F f) {
    if (a.io_dt == kSrcF32) {
        f([&](int64_t i) {
            return *reinterpret_cast<const float4*>(static_cast<const float*>(a.q) + i);
        });
    } else {
        const uint32_t half_mask = a.io_dt == kSrcF16 ? ~0u : 0u;
        f([&, half_mask](int64_t i) { return load4_16(a.q, i, half_mask); });
    }
}
__device__ __forceinline__ uint16_t round16(float x, int dt) {
    return dt == kSrcBF16 ? __builtin_bit_cast(uint16_t, (__bf16)x)
                          : __builtin_bit_cast(uint16_t, (_Float16)x);
}
__device__ __forceinline__ void store4_as(void* p, int64_t i, float4 x, int dt) {
    if (dt == kSrcF32) {
        *reinterpret_cast<float4*>(static_cast<float*>(p) + i) = x;
    } else {
        const uint32_t lo = round16(x.x, dt) | (uint32_t)round16(x.y, dt) << 16;
        const uint32_t hi = round16(x.z, dt) | (uint32_t)round16(x.w, dt) << 16;
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p) + i) = make_uint2(lo, hi);
    }
}

// Piece operands of 8 fp32 values.
template <int NP>
__device__ __forceinline__ void split8(const float* x, u32x4_t* p, SplitConsts k) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t h, m, lo;
        if constexpr (NP == 3) {
            split3_pair(x[2 * j], x[2 * j + 1], h, m, lo, k);
            p[2][j] = lo;
            p[1][j] = m;
        } else if constexpr (NP == 2) {
            split_pair(x[2 * j], x[2 * j + 1], h, m, k);
            p[1][j] = m;
        } else {
            h = pack_bf16x2(x[2 * j], x[2 * j + 1]);
        }
        p[0][j] = h;
    }
}

// The middles of packed values: row m of their operand tile is a block of 32
// channels (which share a value group).
__device__ __forceinline__ constexpr int middle_block(int m, int D) {
    return D > 128 ? m % 8 : m % 4 % (D / 32);
}
// Up to four blocks: the same stacked in one operand, piece m / 4 in row m, the
// last four rows ones, whose sum is the normaliser's: half of the products, and
// one tile to keep in LDS, but the fold crosses lanes.
__device__ __forceinline__ u32x4_t middle_stack(const float* mid, int lane, SplitConsts k) {
    u32x4_t p[3], z;
    split8<3>(mid, p, k);
    const int i = lane % 16 / 4;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        z[c] = i == 0 ? p[0][c] : i == 1 ? p[1][c] : i == 2 ? p[2][c] : 0x3f803f80u;
    return z;
}

// acc[rt] += (sum of A pieces) * (sum of B pieces of rt): the products of
// pieces i and j with i + j < max(NA, NB), smallest first (LAST 1: all but the
// product of the first pieces).
template <int NA, int NB, int RT, int LAST = 0, class B>
__device__ __forceinline__ void mul_pieces(f32x4_t (&acc)[RT], const bf16x8_t* A, const B& b_of) {
    constexpr int N = NA > NB ? NA : NB;
#pragma unroll
    for (int d = N - 1; d >= LAST; --d) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (d - j < 0 || d - j >= NA) continue;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma(A[d - j], b_of(rt, j), acc[rt]);
        }
    }
}

// A 16-bit ring element (in bits 15:0) widened: fp16 where half_mask is all
// ones, bf16 where it is 0 (see load4_16).
__device__ __forceinline__ float widen16(uint32_t h, uint32_t half_mask) {
    const uint32_t f = __float_as_uint((float)__builtin_bit_cast(_Float16, (uint16_t)h));
    return __uint_as_float((f & half_mask) | ((h << 16) & ~half_mask));
}
template <bool R16>
__device__ __forceinline__ uint32_t ring_word(gptr p, uint32_t off) {
    if constexpr (R16) return gload<uint16_t>(p, off);
    else return gload<uint32_t>(p, off);
}

// Ring slot of window token t (clamped to the window: tokens past its end
// repeat the last one and take no weight).
__device__ __forceinline__ int window_slot(const RowsLaunch& a, int t) {
    const int s = a.res_start + min(t, a.res_len - 1);
    return s >= a.Rcap ? s - a.Rcap : s;
}

// Whether some of the wave's query values of rows row0 + 16 rt + l % 16 are not
// bf16 (they take three pieces).
template <int D, int RT>
__device__ __forceinline__ bool wide_queries(const RowsLaunch& a, int row0, int b, int kvh) {
    const int lane = threadIdx.x % kWave;
    uint32_t low = 0;
    with_query(a, [&](auto load) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int r = min(row0 + 16 * rt + lane % 16, a.rows - 1);
        const int64_t q = query_offset(a, b, kvh, r) + 8 * (lane / 16);
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 x = load(q + 32 * ks + 4 * j);
                low |= __float_as_uint(x.x) | __float_as_uint(x.y) | __float_as_uint(x.z) |
                       __float_as_uint(x.w);
            }
        }
    }
    });
    return __builtin_amdgcn_ballot_w64((low & 0xffffu) != 0) != 0;
}

// A wave's RT tiles of 16 query rows: operands, softmax state and output.
// STACKED: the middles' pieces lie in one operand (middle_stack).
template <int D, int RT, int NQ, bool STACKED>
struct Rows {
    static constexpr int KS = D / 32, NBV = D / 16;
    // Three pieces of two tiles do not fit the registers: they lie in LDS, once
    // for the waves of a workgroup that holds the same rows in all of them.
    static constexpr bool Q_LDS = RT * NQ > 3;
    static constexpr int Q_BYTES = RT * KS * NQ * kTile;
    bf16x8_t qf[Q_LDS ? 1 : RT][Q_LDS ? 1 : KS][NQ];
    unsigned char* ql;
    f32x4_t O[RT][NBV];
    f32x4_t Z[RT];                  // weighted middles (STACKED: and weights)
    float m[RT], l[RT];
    int vis[RT];                    // window tokens the lane's row sees
    float qs;                       // |softmax scale * log2 e| (its sign is in the query)
    SplitConsts spc;
    bool bad = false;               // a window sum of this lane came out NaN

    // rows row0 .. (those past the end repeat the last; they are not stored)
    // q_lds (Q_LDS): Q_BYTES of LDS, which the workgroup may read after a barrier.
    __device__ __forceinline__ void init(const RowsLaunch& a, int row0, int b, int kvh,
                                         unsigned char* q_lds = nullptr) {
        const int lane = threadIdx.x % kWave, col = lane % 16, gq = lane / 16;
        ql = q_lds + lane * 16;
        spc = split_consts();
        qs = fabsf(a.qscale);
        const float sign = a.qscale < 0.f ? -1.f : 1.f;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int r = min(row0 + 16 * rt + col, a.rows - 1);
            vis[rt] = min(a.vis0 + r / a.hg, a.res_len);
            // (the lowest finite value: a score of -inf then takes no weight
            // also where it comes first, and any finite one moves it)
            m[rt] = -FLT_MAX;
            l[rt] = 0.f;
            Z[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int nb = 0; nb < NBV; ++nb) O[rt][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        with_query(a, [&](auto load) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int r = min(row0 + 16 * rt + col, a.rows - 1);
            const int64_t q = query_offset(a, b, kvh, r) + 8 * gq;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const float4 x0 = load(q + 32 * ks), x1 = load(q + 32 * ks + 4);
                const float x[8] = {x0.x * sign, x0.y * sign, x0.z * sign, x0.w * sign,
                                    x1.x * sign, x1.y * sign, x1.z * sign, x1.w * sign};
                u32x4_t p[3];
                split8<NQ>(x, p, spc);
#pragma unroll
                for (int i = 0; i < NQ; ++i) {
                    if constexpr (Q_LDS) *q_at(rt, ks, i) = __builtin_bit_cast(bf16x8_t, p[i]);
                    else qf[rt][ks][i] = __builtin_bit_cast(bf16x8_t, p[i]);
                }
            }
        }
        });
    }
    __device__ __forceinline__ bf16x8_t* q_at(int rt, int ks, int i) const {
        return reinterpret_cast<bf16x8_t*>(ql + ((rt * KS + ks) * NQ + i) * kTile);
    }
    __device__ __forceinline__ void query(bf16x8_t (&q)[RT][NQ], int ks) const {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                if constexpr (Q_LDS) q[rt][i] = *q_at(rt, ks, i);
                else q[rt][i] = qf[rt][ks][i];
            }
        }
    }

    // s[rt] += key tile (kKP pieces) x query at k-step ks
    __device__ __forceinline__ void keys(f32x4_t (&s)[RT], const bf16x8_t* kf, int ks) {
        bf16x8_t q[RT][NQ];
        query(q, ks);
        mul_pieces<kKP, NQ, RT>(s, kf, [&](int rt, int j) { return q[rt][j]; });
    }
    // The same for the window's fp32 keys, the small products in a sum of their
    // own: s then rounds once per k-step at its full size, as plain fp32 sums
    // over that many channels at most do.
    __device__ __forceinline__ void window_keys(f32x4_t (&s)[RT], f32x4_t (&small)[RT],
                                                const bf16x8_t* kf, int ks) {
        bf16x8_t q[RT][NQ];
        query(q, ks);
        mul_pieces<kKP, NQ, RT, 1>(small, kf, [&](int rt, int j) { return q[rt][j]; });
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) s[rt] = mfma(kf[0], q[rt][0], s[rt]);
    }

    // Online softmax of a unit's scores s[nb][rt] (unscaled), leaving the
    // weights in p.  Score i of tile nb is the unit's token 4gq + 16nb + i.
    // `hid`: bit t hides token t from every row; WIN: the unit is window
    // tokens t0.., of which row tile rt sees those below vis.
    template <bool WIN>
    __device__ __forceinline__ void softmax(const f32x4_t (&s)[2][RT], uint32_t hid, int t0,
                                            float (&p)[RT][8]) {
        const int gq = (threadIdx.x % kWave) / 16;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = s[i / 4][rt][i % 4];
            uint32_t off = 0;                  // bit i: score i takes no weight
            if (WIN || hid) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int t = 4 * gq + 16 * (i / 4) + i % 4;
                    off |= ((hid >> t) & 1u) << i;
                    if (WIN) off |= t >= vis[rt] - t0 ? 1u << i : 0u;
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = (off >> i) & 1u ? -INFINITY : x[i];
            }
            if (WIN) {
#pragma unroll
                for (int i = 0; i < 8; ++i) bad |= x[i] != x[i];
            }
            float top = x[0];
#pragma unroll
            for (int i = 1; i < 8; ++i) top = fmaxf(top, x[i]);
            top *= qs;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(top > m[rt] + kMoveMax) != 0, 0)) {
                const float cm = row4_max(top);
                if (cm > m[rt] + kMoveMax) {
                    const float f = exp2_fast(m[rt] - cm);
                    m[rt] = cm;
                    l[rt] *= f;
                    Z[rt] *= f;
#pragma unroll
                    for (int nb = 0; nb < NBV; ++nb) O[rt][nb] *= f;
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) p[rt][i] = exp2_fast(fmaf(x[i], qs, -m[rt]));
            if (WIN || hid) {                  // (0 also while the maximum is the lowest)
#pragma unroll
                for (int i = 0; i < 8; ++i) p[rt][i] = (off >> i) & 1u ? 0.f : p[rt][i];
            }
            if (WIN || !STACKED) {
                float sum = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) sum += p[rt][i];
                l[rt] += sum;
            }
        }
    }
    // The weights as operand pieces.
    template <bool WIN>
    __device__ __forceinline__ void weights(const f32x4_t (&s)[2][RT], uint32_t hid, int t0,
                                            bf16x8_t (&pf)[RT][kPP]) {
        float p[RT][8];
        softmax<WIN>(s, hid, t0, p);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            u32x4_t w[3];
            split8<kPP>(p[rt], w, spc);
#pragma unroll
            for (int i = 0; i < kPP; ++i) pf[rt][i] = __builtin_bit_cast(bf16x8_t, w[i]);
        }
    }
    // Z += middles x weights, rounded once per unit.
    static constexpr int MID_TILES = STACKED ? 1 : kPP, MID_PRODUCTS = (STACKED ? 3 : 6) * RT;
    __device__ __forceinline__ void middles(const u32x4_t* zt, const bf16x8_t (&pf)[RT][kPP]) {
        f32x4_t z[RT];
        bf16x8_t zf[MID_TILES];
#pragma unroll
        for (int i = 0; i < MID_TILES; ++i) zf[i] = __builtin_bit_cast(bf16x8_t, zt[i]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) z[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        mul_pieces<MID_TILES, kPP, RT>(z, zf, [&](int rt, int j) { return pf[rt][j]; });
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) Z[rt] += z[rt];
    }
    // O += Z (and l), after the packed units: the lane's Z[.][i] is row 4 gq + i.
    __device__ __forceinline__ void fold_middles() {
        const int gq = (threadIdx.x % kWave) / 16;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if constexpr (STACKED) l[rt] += gq == 3 ? Z[rt][0] : 0.f;
#pragma unroll
            for (int w = 0; w < KS; ++w) {
                float x = Z[rt][w % 4];
                if constexpr (STACKED) {
                    x = row4_sum(gq == 3 ? 0.f : x);
                } else if constexpr (KS > 4) {         // half of the blocks are 16 lanes away
                    const float other = __shfl_xor(x, 16);
                    x = w / 4 == gq % 2 ? x : other;
                }
                O[rt][2 * w] += x;
                O[rt][2 * w + 1] += x;
            }
            Z[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }

    // O[.][nb] += value tile nb (VP pieces) x weights.  A window unit's sum is
    // formed apart and rounds O once.
    template <int VP>
    __device__ __forceinline__ void values(const bf16x8_t* vf, const bf16x8_t (&pf)[RT][kPP], int nb) {
        constexpr bool WIN = VP == kVPWin;
        f32x4_t o[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) o[rt] = WIN ? f32x4_t{0.f, 0.f, 0.f, 0.f} : O[rt][nb];
        mul_pieces<VP, VP, RT>(o, vf, [&](int rt, int j) { return pf[rt][j]; });
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            O[rt][nb] = WIN ? O[rt][nb] + o[rt] : o[rt];
            if (WIN) {
#pragma unroll
                for (int i = 0; i < 4; ++i) bad |= o[rt][i] != o[rt][i];
            }
        }
    }

    // A window unit (tokens t0 ..) in plain fp32 straight from the ring: dot
    // products with a quarter of the channels per lane, four lanes per row, then
    // the lane's channels' weighted sums over the tokens that the row sees.
    template <bool R16>
    __device__ __forceinline__ void plain_unit(const RowsLaunch& a, int64_t bh, int b, int kvh,
                                               int row0, uint32_t hid, int t0) {
        static_assert(RT == 1, "a row tile at a time");
        const int lane = threadIdx.x % kWave, col = lane % 16, gq = lane / 16;
        const float sign = a.qscale < 0.f ? -1.f : 1.f;
        const uint32_t half_mask = a.res_dt == kSrcF16 ? ~0u : 0u;
        auto ring4 = [&](const void* p, int64_t i) {
            if constexpr (R16) return load4_16(p, i, half_mask);
            else return load4_vec<kSrcF32>(p, i);
        };
        float4 q[D / 16];
        with_query(a, [&](auto load) {
            const int64_t at = query_offset(a, b, kvh, min(row0 + col, a.rows - 1)) + 4 * gq;
#pragma unroll
            for (int j = 0; j < D / 16; ++j) q[j] = load(at + 16 * j);
        });
        f32x4_t s[2][RT];
#pragma unroll 2
        for (int t = 0; t < kUnit; ++t) {
            const int64_t k = (bh * a.Rcap + window_slot(a, t0 + t)) * D + 4 * gq;
            float4 y[D / 16];
#pragma unroll
            for (int j = 0; j < D / 16; ++j) y[j] = ring4(a.k_res, k + 16 * j);
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < D / 16; ++j) {
                sum = fmaf(q[j].x, y[j].x, sum);
                sum = fmaf(q[j].y, y[j].y, sum);
                sum = fmaf(q[j].z, y[j].z, sum);
                sum = fmaf(q[j].w, y[j].w, sum);
            }
            sum = row4_sum(sum) * sign;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (t == 4 * gq + 16 * (i / 4) + i % 4) s[i / 4][0][i % 4] = sum;
        }
        float p[RT][8];
        softmax<true>(s, hid, t0, p);
#pragma unroll 2
        for (int t = 0; t < kUnit; ++t) {
            const int64_t v = (bh * a.Rcap + window_slot(a, t0 + t)) * D + 4 * gq;
            float4 y[NBV];
#pragma unroll
            for (int nb = 0; nb < NBV; ++nb) y[nb] = ring4(a.v_res, v + 16 * nb);
            float w = 0.f;                     // the token's weight, where it lies
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j == 4 * (t / 16) + t % 4) w = p[0][j];
            w = __shfl(w, 16 * (t % 16 / 4) + col);
            if (((hid >> t) & 1u) || t >= vis[0] - t0) continue;
#pragma unroll
            for (int nb = 0; nb < NBV; ++nb) {
                O[0][nb][0] = fmaf(w, y[nb].x, O[0][nb][0]);
                O[0][nb][1] = fmaf(w, y[nb].y, O[0][nb][1]);
                O[0][nb][2] = fmaf(w, y[nb].z, O[0][nb][2]);
                O[0][nb][3] = fmaf(w, y[nb].w, O[0][nb][3]);
            }
        }
    }
};

// The unnormalised state of row r -> its partial, or the output when the
// context has one split (a row that sees no position gives 0).
struct RowDst {
    void* p;
    int64_t at;
    int dt;
    float f;
    __device__ __forceinline__ void store4(int d, float x, float y, float z, float w) const {
        store4_as(p, at + d, make_float4(x * f, y * f, z * f, w * f), dt);
    }
};
__device__ __forceinline__ RowDst row_dst(const RowsLaunch& a, int b, int kvh, int64_t bh, int r,
                                          int split, float m, float l, bool first) {
    if (a.n_splits == 1)
        return {a.out, out_offset(a, b, kvh, r), a.io_dt, l > 0.f || l != l ? 1.f / l : 0.f};
    const int64_t row = (bh * a.rows + r) * a.n_splits + split;
    if (first) {
        a.part_ml[row * 2] = m;
        a.part_ml[row * 2 + 1] = l;
    }
    return {a.part_o, row * a.D, kSrcF32, 1.f};
}

// A workgroup's range of units, and which of a unit's tokens are hidden.
struct Range {
    int n_cu;                      // packed units of the context
    int begin, c_end, end;         // packed units [begin, c_end), then window units [.., end)
    int kv_lo;
    const uint32_t* hid_row;
    int vis_most;                  // window tokens that some row of the workgroup sees

    __device__ __forceinline__ Range(const RowsLaunch& a, int split, int b, int last_row) {
        n_cu = a.n_chunks * (a.G / kUnit);
        // splits are even in weight: a window unit counts kWindowWeight
        const int nu = n_cu, all = a.n_units;
        auto at = [nu, all](int x) {
            return x <= nu ? x : min(nu + (x - nu + kWindowWeight - 1) / kWindowWeight, all);
        };
        begin = at(split * a.weight_per_split);
        end = at((split + 1) * a.weight_per_split);
        c_end = min(end, n_cu);
        kv_lo = __builtin_amdgcn_readfirstlane(a.kv_start ? a.kv_start[b] : 0);
        hid_row = a.hidden ? a.hidden + b * a.hidden_stride : nullptr;
        vis_most = min(a.vis0 + min(last_row, a.rows - 1) / a.hg, a.res_len);
    }
    __device__ __forceinline__ uint32_t hidden(int u) const {       // wave-uniform
        const int n = kv_lo - kUnit * u;
        uint32_t h = n >= kUnit ? ~0u : n > 0 ? (1u << n) - 1u : 0u;
        if (hid_row) h |= hid_row[u];
        return h;
    }
    // one past the last window unit that some row sees
    __device__ __forceinline__ int w_end() const {
        return min(end, n_cu + (vis_most + kUnit - 1) / kUnit);
    }
};

// ---------------------------------------------------------------------------
// Many rows: units expanded into LDS by the whole workgroup.
//
// What bounds it: a wave's step is 102 matrix products (1632 cycles) of two row
// tiles, ~300 vector instructions and 41 KB of LDS reads; two waves per SIMD
// take ~6400 cycles per step, the products 3260 of them (47 % of all SIMD cycles
// with prologue and window), the LDS reads 2600 (each 1 KB operand feeds two row
// tiles).  Also measured for 512 query tokens, before the middles' tile (215 us
// kernel time then): 4 waves with 128 rows and two workgroups per CU 264 us; 4
// waves with four row tiles each (half the LDS reads, one wave per SIMD, 66
// registers spilled) 295 us; a raised priority for half of the waves 224 us.
// ---------------------------------------------------------------------------
template <int D>
struct SharedShape {
    static constexpr int KS = D / 32, NBV = D / 16;
    static constexpr int WAVES = D <= 128 ? 8 : 4, BLOCK = WAVES * kWave;
    // code words of a unit that each wave expands (a word: one lane-word of
    // the key or value operands, two tiles); at head_dim 64 the last four
    // waves have none
    static constexpr int WORDS = 2 * KS / WAVES > 0 ? 2 * KS / WAVES : 1;
    static constexpr int RT = D <= 128 ? 2 : 1;   // most row tiles per wave
    // value tiles are spaced for three pieces where LDS allows (packed values
    // then write a third piece nobody reads, instead of branching)
    static constexpr int VSTR = WORDS > 1 ? 2 : 3;
    static constexpr int K_BYTES = KS * 2 * kKP * kTile;
    // the middles' tile, stacked (at head_dim 256 LDS is full: each wave makes
    // their operands itself)
    static constexpr bool MID_LDS = D <= 128;
    static constexpr int MID = K_BYTES + NBV * VSTR * kTile;
    static constexpr int BUF = MID + (MID_LDS ? kTile : 0);
    static constexpr int LDS = 2 * BUF;
    static_assert(K_BYTES + NBV * kVPWin * kTile <= LDS, "a window unit fits");
};

// Word i of a wave: key word or value word w.  At head_dim 256 a wave has two
// of each, keys first; below, one word.
struct Word {
    bool key;
    int w;
};
// (at head_dim 64 the last four waves have none)
template <int D>
__device__ __forceinline__ bool has_word(int wave) {
    return 2 * (D / 32) >= SharedShape<D>::WAVES || wave < 2 * (D / 32);
}
template <int D>
__device__ __forceinline__ Word word_of(int i, int wave) {
    constexpr int KS = D / 32;
    constexpr int HALF = SharedShape<D>::WORDS / 2;
    if constexpr (HALF > 0) return {i < HALF, wave + SharedShape<D>::WAVES * (i % HALF)};
    return {wave < KS, wave % KS};
}

// Byte offset, in a value operand tile, of row lane % 16's tokens 8 (lane / 16) ..
// + 3 (the next four lie 256 bytes on).
__device__ __forceinline__ uint32_t value_slot(int lane) {
    const int gq = lane / 16;
    return ((2 * (gq % 2)) * 16 + lane % 16) * 16 + 8 * (gq / 2);
}

// Where a thread stores its words' pieces: byte offset in a buffer of (tile 2w,
// piece 0)'s first half, distance of the second half, of the tiles 2w + 1, of
// the pieces (kTile).  Key operands are lane-major.  Value operands: this
// lane's 8 tokens 8(l/16)..+7 of a channel go to the operand slots (g, j) of
// tokens 4g + j%4 + 16(j/4), the order the scores lie in.
template <int D>
struct Dst {
    uint32_t at[SharedShape<D>::WORDS], half[SharedShape<D>::WORDS], tile[SharedShape<D>::WORDS];
    __device__ __forceinline__ Dst(int wave, int lane, int vstr) {
#pragma unroll
        for (int i = 0; i < SharedShape<D>::WORDS; ++i) {
            const Word x = word_of<D>(i, wave);
            at[i] = x.key ? (2 * x.w * kKP) * kTile + lane * 16
                          : SharedShape<D>::K_BYTES + (2 * x.w * vstr) * kTile + value_slot(lane);
            half[i] = x.key ? 8 : 256;
            tile[i] = (x.key ? kKP : vstr) * kTile;
        }
    }
};

// Stores the pieces of one tile's 8 values.
template <int NP>
__device__ __forceinline__ void put_tile(unsigned char* at, uint32_t half, const float* x,
                                         SplitConsts k) {
    u32x4_t p[3];
    split8<NP>(x, p, k);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        *reinterpret_cast<uint2*>(at + i * kTile) = make_uint2(p[i][0], p[i][1]);
        *reinterpret_cast<uint2*>(at + i * kTile + half) = make_uint2(p[i][2], p[i][3]);
    }
}

// A thread's words of a packed unit with the 8 scales and zeros of their 8
// channels (keys) or 8 tokens (values), and where they come from.
template <int D>
struct PackedUnit {
    static constexpr int N = SharedShape<D>::WORDS;
    uint32_t word[N];
    kivi_f4v sc[N][2], zr[N][2];
    // at chunk 0 of the (batch, kv head): wave-uniform bases, bytes per chunk
    // and per second unit of a G = 64 chunk, and this lane's bytes
    gptr code[N], scale[N], zero[N];
    uint32_t code_step[N], code_half[N], meta_step[N], meta_half[N], code_off[N], meta_off[N];

    __device__ __forceinline__ void init(const RowsLaunch& a, int64_t bh, int wave, int lane) {
        const int two = a.G == 64 ? 2 : 1;    // units per chunk
        const int64_t c0 = bh * a.Cmax;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const Word x = word_of<D>(i, wave);
            code_step[i] = a.G * D / 4;
            code_half[i] = x.key ? 4 : D / 8;
            meta_step[i] = 4 * (x.key ? D : D / a.Gv * a.G);
            meta_half[i] = x.key ? 0 : 4 * kUnit;
            code[i] = (gptr)(x.key ? a.k_codes : a.v_codes) + c0 * code_step[i];
            scale[i] = (gptr)(x.key ? a.k_scale : a.v_scale) + c0 * meta_step[i];
            zero[i] = (gptr)(x.key ? a.k_zero : a.v_zero) + c0 * meta_step[i];
            code_off[i] = 4u * (lane * (two * (D / 32)) + (x.key ? x.w * two : x.w));
            meta_off[i] = 4u * ((x.key ? 32 * x.w : 32 * x.w / a.Gv * a.G) + 8 * (lane / 16));
        }
    }
    __device__ __forceinline__ void load(int two, int u) {
        const uint32_t chunk = two ? u >> 1 : u, half = two ? u & 1 : 0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const gptr c = code[i] + (chunk * code_step[i] + half * code_half[i]);
            const uint32_t m = chunk * meta_step[i] + half * meta_half[i];
            word[i] = gload<uint32_t>(c, code_off[i]);
            sc[i][0] = gload<kivi_f4v>(scale[i] + m, meta_off[i]);
            sc[i][1] = gload<kivi_f4v>(scale[i] + m, meta_off[i] + 16);
            zr[i][0] = gload<kivi_f4v>(zero[i] + m, meta_off[i]);
            zr[i][1] = gload<kivi_f4v>(zero[i] + m, meta_off[i] + 16);
        }
    }
    // Value words enter as offsets from the middle of their group's range, c vs -
    // 1.5 vs: call once after load().
    float mid[8];                  // N == 1: the word's middles
    __device__ __forceinline__ void center(int wave) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const bool key = word_of<D>(i, wave).key;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if constexpr (N == 1) mid[c] = fmaf(1.5f, sc[i][c / 4][c % 4], zr[i][c / 4][c % 4]);
                zr[i][c / 4][c % 4] = key ? zr[i][c / 4][c % 4] : -1.5f * sc[i][c / 4][c % 4];
            }
        }
    }
    // N == 1: a value word's rows of the middles' tile.
    __device__ __forceinline__ void put_middles(unsigned char* buf, int wave, int lane,
                                                SplitConsts k) const {
        const Word w = word_of<D>(0, wave);
        if (w.key || !has_word<D>(wave)) return;
        const u32x4_t z = middle_stack(mid, lane, k);
        if (middle_block(lane % 16, D) != w.w) return;
        unsigned char* at = buf + SharedShape<D>::MID + value_slot(lane);
        *reinterpret_cast<uint2*>(at) = make_uint2(z[0], z[1]);
        *reinterpret_cast<uint2*>(at + 256) = make_uint2(z[2], z[3]);
    }
    // Expands tile m of every word into buffer `buf`.
    template <int M>
    __device__ __forceinline__ void expand(unsigned char* buf, const Dst<D>& d, int wave,
                                           SplitConsts k) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const Word w = word_of<D>(i, wave);
            const float s[8] = {sc[i][0].x, sc[i][0].y, sc[i][0].z, sc[i][0].w,
                                sc[i][1].x, sc[i][1].y, sc[i][1].z, sc[i][1].w};
            const float z[8] = {zr[i][0].x, zr[i][0].y, zr[i][0].z, zr[i][0].w,
                                zr[i][1].x, zr[i][1].y, zr[i][1].z, zr[i][1].w};
            float x[8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {     // elements 2c and 2c + 1: bytes M and 2 + M
                const uint32_t y = (word[i] >> (2 * c)) & 0x03030303u;
                x[2 * c] = fmaf((float)((y >> (8 * M)) & 0xffu), s[2 * c], z[2 * c]);
                x[2 * c + 1] = fmaf((float)((y >> (16 + 8 * M)) & 0xffu), s[2 * c + 1],
                                    z[2 * c + 1]);
            }
            unsigned char* at = buf + d.at[i] + M * d.tile[i];
            if constexpr (N > 1) {            // (the kind of word is known)
                if (w.key) put_tile<kKP>(at, d.half[i], x, k);
                else put_tile<kVPChunk>(at, d.half[i], x, k);
            } else if (has_word<D>(wave)) {
                put_tile<kKP>(at, d.half[i], x, k);
            }
        }
    }
};

// The middles of the lane's row for the 8 tokens of its operand slots, from
// global memory.
template <int D>
struct Middles {
    kivi_f4v sc[2], zr[2];

    __device__ __forceinline__ void load(const RowsLaunch& a, int64_t bh, int u, int lane) {
        const int two = a.G == 64 ? 2 : 1, ng = D / a.Gv;
        const int chunk = two == 2 ? u >> 1 : u, half = two == 2 ? u & 1 : 0;
        const int64_t at = (bh * a.Cmax + chunk) * ng * a.G + kUnit * half;
        const uint32_t off =
            4u * (32 * middle_block(lane % 16, D) / a.Gv * a.G + 4 * (lane / 16));
        const gptr s = (gptr)(a.v_scale + at), z = (gptr)(a.v_zero + at);
        sc[0] = gload<kivi_f4v>(s, off);
        sc[1] = gload<kivi_f4v>(s, off + 64);
        zr[0] = gload<kivi_f4v>(z, off);
        zr[1] = gload<kivi_f4v>(z, off + 64);
    }
    __device__ __forceinline__ void operands(u32x4_t* zf, SplitConsts k) const {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = fmaf(1.5f, sc[j / 4][j % 4], zr[j / 4][j % 4]);
        split8<kPP>(x, zf, k);
    }
};

// A thread's words of a window unit, as the ring holds them (widened when
// they are expanded, so that nothing waits for the loads before).
template <int D, bool R16>
struct WindowUnit {
    static constexpr int N = SharedShape<D>::WORDS, E = R16 ? 2 : 4;
    uint32_t raw[N][16];

    __device__ __forceinline__ void load(const RowsLaunch& a, int64_t bh, int t0, int wave,
                                         int lane) {
        const int gq = lane / 16, col = lane % 16;
        const int64_t base = bh * a.Rcap * D * E;
        const gptr kr = (gptr)a.k_res + base, vr = (gptr)a.v_res + base;
        if (!has_word<D>(wave)) return;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const Word w = word_of<D>(i, wave);
            if (w.key) {
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const uint32_t o = E * ((uint32_t)window_slot(a, t0 + 16 * m + col) * D +
                                            32 * w.w + 8 * gq);
#pragma unroll
                    for (int q = 0; q < E / 2; ++q) {
                        const u32x4_t x = gload<u32x4_t>(kr, o + 16 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) raw[i][8 * m + 4 * q + e] = x[e];
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t o = E * ((uint32_t)window_slot(a, t0 + 8 * gq + j) * D +
                                            32 * w.w + col);
#pragma unroll
                    for (int m = 0; m < 2; ++m) raw[i][8 * m + j] = ring_word<R16>(vr, o + 16 * E * m);
                }
            }
        }
    }
    __device__ __forceinline__ void expand(unsigned char* buf, const Dst<D>& d, int wave,
                                           uint32_t half_mask, SplitConsts k) const {
        if (!has_word<D>(wave)) return;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const bool key = word_of<D>(i, wave).key;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (!R16) x[j] = __uint_as_float(raw[i][8 * m + j]);
                    else if (key) x[j] = widen16((raw[i][8 * m + j / 2] >> (16 * (j % 2))) & 0xffffu, half_mask);
                    else x[j] = widen16(raw[i][8 * m + j], half_mask);
                }
                put_tile<3>(buf + d.at[i] + m * d.tile[i], d.half[i], x, k);
            }
        }
    }
};

// Between two operand tiles' products: the LDS reads and the products keep their
// order, everything else may cross.  The reads run two tiles ahead of the
// products; left to itself the compiler reads a tile right before its products
// and waits out the LDS latency each time.
__device__ __forceinline__ void keep_order() {
    constexpr int kValu = 0x2, kSalu = 0x4, kVmem = 0x10 | 0x20 | 0x40, kDsWrite = 0x200,
                  kTrans = 0x400;
    __builtin_amdgcn_sched_barrier(kValu | kSalu | kVmem | kDsWrite | kTrans);
}

// Returns whether a window sum of this thread came out NaN.  PLAIN: the window
// in plain fp32.
template <int D, int RT, int NQ, bool R16, bool PLAIN>
__device__ bool walk_shared(const RowsLaunch& a, unsigned char* smem, const Range& rg, int row0,
                            int64_t bh, int b, int kvh, int split) {
    using S = SharedShape<D>;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool active = row0 < a.rows;         // wave-uniform
    Rows<D, RT, NQ, S::MID_LDS> rows;
    rows.init(a, row0, b, kvh);

    // One unit from LDS buffer `buf`; after_k and after_v run behind the reads
    // of the key and of the value tiles: the expansion of the next unit, whose
    // vector work then sits among this unit's matrix products.
    auto use_unit = [&](const unsigned char* buf, uint32_t hid, int t0, auto win_c, int vstr,
                        const Middles<D>& mid, auto&& after_k, auto&& after_v) {
        constexpr bool WIN = decltype(win_c)::value;
        constexpr int VP = WIN ? kVPWin : kVPChunk;
        f32x4_t s[2][RT], small[2][RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            s[0][rt] = s[1][rt] = small[0][rt] = small[1][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        constexpr int AHEAD = D > 128 ? 1 : 2;
        bf16x8_t kf[2 * S::KS][kKP];
        auto read_keys = [&](int t) {
#pragma unroll
            for (int p = 0; p < kKP; ++p)
                kf[t][p] = *reinterpret_cast<const bf16x8_t*>(buf + (t * kKP + p) * kTile + lane * 16);
        };
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) read_keys(t);
        keep_order();
#pragma unroll
        for (int t = 0; t < 2 * S::KS; ++t) {
            if (t + AHEAD < 2 * S::KS) read_keys(t + AHEAD);
            if constexpr (WIN) rows.window_keys(s[t % 2], small[t % 2], kf[t], t / 2);
            else rows.keys(s[t % 2], kf[t], t / 2);
            keep_order();
        }
        if constexpr (WIN) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                s[0][rt] += small[0][rt];
                s[1][rt] += small[1][rt];
            }
        }
        after_k();
        bf16x8_t pf[RT][kPP];
        rows.template weights<WIN>(s, hid, t0, pf);
        bf16x8_t vf[S::NBV][VP];
        auto read_values = [&](int nb) {
#pragma unroll
            for (int p = 0; p < VP; ++p)
                vf[nb][p] = *reinterpret_cast<const bf16x8_t*>(buf + S::K_BYTES +
                                                               (nb * vstr + p) * kTile + lane * 16);
        };
        if constexpr (!WIN) {
            u32x4_t zf[decltype(rows)::MID_TILES];
            if constexpr (S::MID_LDS)
                zf[0] = *reinterpret_cast<const u32x4_t*>(buf + S::MID + lane * 16);
            else
                mid.operands(zf, rows.spc);
#pragma unroll
            for (int nb = 0; nb < AHEAD; ++nb) read_values(nb);
            keep_order();
            rows.middles(zf, pf);
        } else {
#pragma unroll
            for (int nb = 0; nb < AHEAD; ++nb) read_values(nb);
        }
        keep_order();
#pragma unroll
        for (int nb = 0; nb < S::NBV; ++nb) {
            if (nb + AHEAD < S::NBV) read_values(nb + AHEAD);
            rows.template values<VP>(vf[nb], pf, nb);
            keep_order();
        }
        after_v();
    };

    if (rg.begin < rg.c_end) {
        PackedUnit<D> unit;
        const Dst<D> dst(wave, lane, S::VSTR);
        const int two = a.G == 64;
        unit.init(a, bh, wave, lane);
        unit.load(two, rg.begin);
        lds_barrier();                         // an earlier walk has read its last unit
        unit.center(wave);
        unit.template expand<0>(smem, dst, wave, rows.spc);
        unit.template expand<1>(smem, dst, wave, rows.spc);
        if constexpr (S::MID_LDS) unit.put_middles(smem, wave, lane, rows.spc);
        unit.load(two, min(rg.begin + 1, rg.c_end - 1));
        for (int u = rg.begin; u < rg.c_end; ++u) {
            const uint32_t hid = rg.hidden(u);
            unsigned char* cur = smem + ((u - rg.begin) & 1) * S::BUF;
            unsigned char* nxt = smem + ((u - rg.begin + 1) & 1) * S::BUF;
            Middles<D> mid;
            if constexpr (!S::MID_LDS) mid.load(a, bh, u, lane);
            lds_barrier();                     // cur is written, nxt has been read
            auto first = [&] {
                unit.center(wave);
                unit.template expand<0>(nxt, dst, wave, rows.spc);
            };
            auto second = [&] {
                unit.template expand<1>(nxt, dst, wave, rows.spc);
                if constexpr (!S::MID_LDS) unit.load(two, min(u + 2, rg.c_end - 1));
            };
            if (active && hid != ~0u) {
                use_unit(cur, hid, 0, BoolC<false>{}, S::VSTR, mid, first, second);
            } else {
                // (as a loop: as plain code the compiler moves what both arms
                // share above the branch, where it waits for unit's loads
                // before any product: 36 rows over 2K, B=16 68 us, so 61)
                int once = 1;
                asm volatile("" : "+s"(once));
#pragma unroll 1
                for (; once; --once) {
                    first();
                    second();
                }
            }
            if constexpr (S::MID_LDS) {        // (a branch: it would break the order above)
                unit.put_middles(nxt, wave, lane, rows.spc);
                unit.load(two, min(u + 2, rg.c_end - 1));
            }
        }
        rows.fold_middles();
    }
    const int w_begin = max(rg.begin, rg.n_cu), w_end = rg.w_end();
    if constexpr (PLAIN) {
        for (int u = w_begin; active && u < w_end; ++u)
            rows.template plain_unit<R16>(a, bh, b, kvh, row0, rg.hidden(u), kUnit * (u - rg.n_cu));
    } else if (w_begin < w_end) {
        WindowUnit<D, R16> unit;
        const uint32_t half_mask = a.res_dt == kSrcF16 ? ~0u : 0u;
        const Dst<D> dst(wave, lane, kVPWin);
        unit.load(a, bh, kUnit * (w_begin - rg.n_cu), wave, lane);
        for (int u = w_begin; u < w_end; ++u) {
            const int t0 = kUnit * (u - rg.n_cu);
            const uint32_t hid = rg.hidden(u);
            lds_barrier();                     // the previous unit has been read
            unit.expand(smem, dst, wave, half_mask, rows.spc);
            unit.load(a, bh, t0 + kUnit, wave, lane);
            lds_barrier();
            if (active) use_unit(smem, hid, t0, BoolC<true>{}, kVPWin, {}, [] {}, [] {});
        }
    }

    if (!active) return false;
    const int gq = lane / 16;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float l = row4_sum(rows.l[rt]);
        const int r = row0 + 16 * rt + lane % 16;
        if (r >= a.rows) continue;
        const RowDst d = row_dst(a, b, kvh, bh, r, split, rows.m[rt], l, gq == 0);
#pragma unroll
        for (int nb = 0; nb < S::NBV; ++nb) {
            const f32x4_t o = rows.O[rt][nb];
            d.store4(16 * nb + 4 * gq, o[0], o[1], o[2], o[3]);
        }
    }
    return rows.bad;
}

template <int D, int RT, bool R16>
__global__ __launch_bounds__(SharedShape<D>::BLOCK) __attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1)))
void attn_rows_shared_kernel(RowsLaunch a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int split = blockIdx.x % a.n_splits, rblock = blockIdx.x / a.n_splits;
    const int kvh = blockIdx.y, b = blockIdx.z;
    const int64_t bh = (int64_t)b * a.Hkv + kvh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int block0 = rblock * a.block_rows, row0 = block0 + wave * 16 * RT;
    const Range rg(a, split, b, block0 + a.block_rows - 1);
    // OR of a value of each wave (before or after the units take the space)
    int* word = reinterpret_cast<int*>(smem);
    auto any_wave = [&](int mine) {
        lds_barrier();
        if (threadIdx.x % kWave == 0) word[wave] = mine;
        lds_barrier();
        int x = 0;
#pragma unroll
        for (int w = 0; w < SharedShape<D>::WAVES; ++w) x |= word[w];
        lds_barrier();
        return __builtin_amdgcn_readfirstlane(x);
    };
    // What the workgroup's queries need (uniform: both walks hold workgroup
    // barriers).
    bool bad = false;
    if (!any_wave(wide_queries<D, RT>(a, row0, b, kvh))) {
        bad = walk_shared<D, RT, 1, R16, false>(a, smem, rg, row0, bh, b, kvh, split);
    } else {
        // three query pieces: one row tile at a time (the pieces of two do not
        // fit the registers)
        for (int rt = 0; rt < RT && block0 + 16 * rt < a.rows; ++rt)
            bad |= walk_shared<D, 1, 3, R16, false>(a, smem, rg, row0 + 16 * rt, bh, b, kvh, split);
    }
    if (__builtin_expect(any_wave(__builtin_amdgcn_ballot_w64(bad) != 0), 0)) {
        __syncthreads();                       // the first results are written
        for (int rt = 0; rt < RT && block0 + 16 * rt < a.rows; ++rt)
            walk_shared<D, 1, 3, R16, true>(a, smem, rg, row0 + 16 * rt, bh, b, kvh, split);
    }
}

// ---------------------------------------------------------------------------
// Few rows: each wave expands units of its own into its registers, with no
// barrier and no LDS traffic but the scales.
//
// What bounds it: the expansion's vector work, ~1000 instructions per unit
// (4-5.5 cycles each) against 1728 cycles of matrix products for two row tiles
// (17 % of all SIMD cycles); two workgroups per CU gain little over one (39
// against 42 us at B=8, 5 query tokens over 4K, with ~100 instructions less).
// ---------------------------------------------------------------------------
constexpr int kWaveWaves = 4, kWaveBlock = kWaveWaves * kWave;

template <int D>
struct WaveShape {
    static constexpr int KS = D / 32, NBV = D / 16;
    static constexpr int RT = D <= 128 ? 2 : 1;
    // a wave's staged scales and zeros: keys [2][D], values [2][D/Gv][32] (at
    // most [2][D])
    static constexpr int META = 4 * D * 4;
    static constexpr int NMETA = (D + kWave - 1) / kWave;       // float4s per lane
    // one wave's state of 16 RT rows: o [16 RT][D], m and l
    static constexpr int STATE = 16 * RT * (D + 2) * 4;
    static constexpr int LDS = kWaveWaves * (STATE > META ? STATE : META);
};

// A lane's loads of one packed unit.  A key word is used as it lies (two
// tiles).  A lane's value operand holds tokens 4gq..+3 and 16+4gq..+3, half
// of what the words of lane groups gq/2 (va) and 2 + gq/2 (vb) hold.
template <int D>
struct WaveUnit {
    static constexpr int KS = D / 32;
    uint32_t k[KS], va[KS], vb[KS];
    kivi_f4v meta[WaveShape<D>::NMETA];

    __device__ __forceinline__ void load_codes(const RowsLaunch& a, int64_t bh, int u, int lane) {
        const int two = a.G == 64 ? 2 : 1;
        const int chunk = two == 2 ? u >> 1 : u, half = two == 2 ? u & 1 : 0;
        const int64_t c0 = (bh * a.Cmax + chunk) * (a.G * D / 4);
        const uint32_t src = 16 * (lane / 32) + lane % 16;
        const uint32_t np = two * KS;
        const gptr kc = (gptr)a.k_codes + c0 + 4 * half, vc = (gptr)a.v_codes + c0 + 4 * half * KS;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            k[ks] = gload<uint32_t>(kc, 4u * (lane * np + ks * two));
            va[ks] = gload<uint32_t>(vc, 4u * (src * np + ks));
            vb[ks] = gload<uint32_t>(vc, 4u * ((src + 32) * np + ks));
        }
    }
    // float4 e of [ks | kz | vs of the unit | vz of the unit]
    __device__ __forceinline__ void load_meta(const RowsLaunch& a, int64_t bh, int u, int lane,
                                              int ng) {
        const int two = a.G == 64 ? 2 : 1;
        const int chunk = two == 2 ? u >> 1 : u, half = two == 2 ? u & 1 : 0;
        const int64_t cid = bh * a.Cmax + chunk;
        const int kq = D / 4, vq = ng * 8;
#pragma unroll
        for (int i = 0; i < WaveShape<D>::NMETA; ++i) {
            const int e = min(lane + kWave * i, 2 * kq + 2 * vq - 1);
            gptr p;
            if (e < 2 * kq) {
                p = (gptr)(e < kq ? a.k_scale + 4 * e : a.k_zero + 4 * (e - kq)) + 4 * cid * D;
            } else {
                const int f = e - 2 * kq, g = f < vq ? f : f - vq;
                p = (gptr)(f < vq ? a.v_scale : a.v_zero) +
                    4 * ((cid * ng + g / 8) * a.G + kUnit * half + 4 * (g % 8));
            }
            meta[i] = gload<kivi_f4v>(p, 0);
        }
    }
    __device__ __forceinline__ void stage_meta(float* mt, int lane, int ng) const {
        const int n = D / 2 + 16 * ng;
#pragma unroll
        for (int i = 0; i < WaveShape<D>::NMETA; ++i) {
            // (a lane past the end holds the last float4 and writes it again)
            const int e = min(lane + kWave * i, n - 1);
            reinterpret_cast<kivi_f4v*>(mt)[e] = meta[i];
        }
    }
};

// N elements, from 0 on, of both tiles of a code word.
template <int N>
__device__ __forceinline__ void expand_word(uint32_t word, const float* s, const float* z, float* x0,
                                            float* x1) {
#pragma unroll
    for (int c = 0; c < N / 2; ++c) {
        // bytes: tile 0 element 2c, tile 1 element 2c, tile 0 element 2c+1, tile 1 ...
        const uint32_t y = (word >> (2 * c)) & 0x03030303u;
        x0[2 * c] = fmaf((float)(y & 0xffu), s[2 * c], z[2 * c]);
        x1[2 * c] = fmaf((float)((y >> 8) & 0xffu), s[2 * c], z[2 * c]);
        x0[2 * c + 1] = fmaf((float)((y >> 16) & 0xffu), s[2 * c + 1], z[2 * c + 1]);
        x1[2 * c + 1] = fmaf((float)(y >> 24), s[2 * c + 1], z[2 * c + 1]);
    }
}

__device__ __forceinline__ void read4(const float* p, float* x) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
}

template <int NP>
__device__ __forceinline__ void operands8(const float* x, bf16x8_t* f, SplitConsts k) {
    u32x4_t p[3];
    split8<NP>(x, p, k);
#pragma unroll
    for (int i = 0; i < NP; ++i) f[i] = __builtin_bit_cast(bf16x8_t, p[i]);
}

template <int D, int RT, int NQ, bool R16, bool PLAIN>
__device__ bool walk_wave(const RowsLaunch& a, unsigned char* smem, const Range& rg, int row0,
                          int64_t bh, int b, int kvh, int split) {
    constexpr int KS = D / 32;
    const int lane = threadIdx.x % kWave, gq = lane / 16, col = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    Rows<D, RT, NQ, false> rows;
    static_assert(!decltype(rows)::Q_LDS ||
                  kWaveWaves * WaveShape<D>::META + decltype(rows)::Q_BYTES <= WaveShape<D>::LDS,
                  "the query's pieces lie behind the staged scales");
    rows.init(a, row0, b, kvh, smem + kWaveWaves * WaveShape<D>::META);   // (by every wave alike)
    if constexpr (decltype(rows)::Q_LDS) lds_barrier();
    const int ng = D / a.Gv;
    float* mt = reinterpret_cast<float*>(smem + wave * WaveShape<D>::META);

    // packed units begin + wave, + 4, ...
    if (rg.begin + wave < rg.c_end) {
        WaveUnit<D> unit;
        unit.load_meta(a, bh, rg.begin + wave, lane, ng);
        unit.load_codes(a, bh, rg.begin + wave, lane);
        const int vshift = 4 * (gq % 2);       // the lane's half of its value words
        for (int u = rg.begin + wave; u < rg.c_end; u += kWaveWaves) {
            const uint32_t hid = rg.hidden(u);
            const int next = min(u + kWaveWaves, rg.c_end - 1);
            wave_sync();                      // the previous unit's reads come first
            unit.stage_meta(mt, lane, ng);
            wave_sync();
            unit.load_meta(a, bh, next, lane, ng);
            f32x4_t s[2][RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s[0][rt] = s[1][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float sc[8], zr[8], x[2][8];
                bf16x8_t kf[kKP];
                const float* p = mt + 32 * ks + 8 * gq;
                read4(p, sc);
                read4(p + 4, sc + 4);
                read4(p + D, zr);
                read4(p + D + 4, zr + 4);
                expand_word<8>(unit.k[ks], sc, zr, x[0], x[1]);
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    operands8<kKP>(x[nb], kf, rows.spc);
                    rows.keys(s[nb], kf, ks);
                }
            }
            bf16x8_t pf[RT][kPP];
            rows.template weights<false>(s, hid, 0, pf);
            {
                float sc[8], x[8];
                u32x4_t zf[kPP];
                const float* p = mt + 2 * D + kUnit * (32 * middle_block(col, D) / a.Gv) + 4 * gq;
                read4(p, sc);
                read4(p + 16, sc + 4);
                read4(p + kUnit * ng, x);
                read4(p + kUnit * ng + 16, x + 4);
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = fmaf(1.5f, sc[j], x[j]);
                split8<kPP>(x, zf, rows.spc);
                rows.middles(zf, pf);
            }
#pragma unroll
            for (int w = 0; w < KS; ++w) {
                float sc[8], zr[8], x[2][8];
                bf16x8_t vf[kVPChunk];
                const float* p = mt + 2 * D + kUnit * (32 * w / a.Gv) + 4 * gq;
                read4(p, sc);
                read4(p + 16, sc + 4);
#pragma unroll
                for (int j = 0; j < 8; ++j) zr[j] = -1.5f * sc[j];
                expand_word<4>(unit.va[w] >> vshift, sc, zr, x[0], x[1]);
                expand_word<4>(unit.vb[w] >> vshift, sc + 4, zr + 4, x[0] + 4, x[1] + 4);
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    operands8<kVPChunk>(x[m], vf, rows.spc);
                    rows.template values<kVPChunk>(vf, pf, 2 * w + m);
                }
            }
            unit.load_codes(a, bh, next, lane);
        }
        rows.fold_middles();
    }
    // window units, dealt in the same turn
    constexpr int E = R16 ? 2 : 4;
    const gptr kr = (gptr)a.k_res + bh * a.Rcap * D * E, vr = (gptr)a.v_res + bh * a.Rcap * D * E;
    const uint32_t half_mask = a.res_dt == kSrcF16 ? ~0u : 0u;
    const int w_begin = max(rg.begin, rg.n_cu), w_end = rg.w_end();
    for (int u = w_begin + (wave + rg.begin + 4 * kWaveWaves - w_begin % kWaveWaves) % kWaveWaves;
         u < w_end; u += kWaveWaves) {
        const int t0 = kUnit * (u - rg.n_cu);
        const uint32_t hid = rg.hidden(u);
        if constexpr (PLAIN) {
            rows.template plain_unit<R16>(a, bh, b, kvh, row0, hid, t0);
            continue;
        }
        // (Key loads run up to four k-steps ahead of their use, and a value tile's
        // are issued before the tile before it is used; left to itself the compiler
        // waits for each load where registers are short.)
        constexpr int AHEAD = KS < 4 ? KS : 4, kNoMemory = 0x1;
        u32x4_t kq[AHEAD][2][E / 2];
        uint32_t ko[2], vo[8];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
            ko[nb] = E * ((uint32_t)window_slot(a, t0 + 16 * nb + col) * D + 8 * gq);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            vo[j] = E * ((uint32_t)window_slot(a, t0 + 4 * gq + 16 * (j / 4) + j % 4) * D + col);
        auto load_keys = [&](int ks) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
                for (int q = 0; q < E / 2; ++q)
                    kq[ks % AHEAD][nb][q] = gload<u32x4_t>(kr, ko[nb] + 32 * E * ks + 16 * q);
            }
        };
        f32x4_t s[2][RT], small[2][RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            s[0][rt] = s[1][rt] = small[0][rt] = small[1][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < AHEAD; ++ks) load_keys(ks);
        __builtin_amdgcn_sched_barrier(kNoMemory);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float x[2][8];
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t d = kq[ks % AHEAD][nb][R16 ? 0 : j / 4][R16 ? j / 2 : j % 4];
                    x[nb][j] = R16 ? widen16((d >> (16 * (j % 2))) & 0xffffu, half_mask)
                                   : __uint_as_float(d);
                }
            }
            if (ks + AHEAD < KS) {
                load_keys(ks + AHEAD);
                __builtin_amdgcn_sched_barrier(kNoMemory);
            }
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                bf16x8_t kf[kKP];
                operands8<kKP>(x[nb], kf, rows.spc);
                rows.window_keys(s[nb], small[nb], kf, ks);
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            s[0][rt] += small[0][rt];
            s[1][rt] += small[1][rt];
        }
        bf16x8_t pf[RT][kPP];
        rows.template weights<true>(s, hid, t0, pf);
        uint32_t vw[2][8];
        auto load_values = [&](int nb) {
#pragma unroll
            for (int j = 0; j < 8; ++j) vw[nb % 2][j] = ring_word<R16>(vr, vo[j] + 16 * E * nb);
        };
        load_values(0);
#pragma unroll
        for (int nb = 0; nb < D / 16; ++nb) {
            float x[8];
            bf16x8_t vf[kVPWin];
            if (nb + 1 < D / 16) load_values(nb + 1);
            __builtin_amdgcn_sched_barrier(kNoMemory);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = R16 ? widen16(vw[nb % 2][j], half_mask) : __uint_as_float(vw[nb % 2][j]);
            operands8<kVPWin>(x, vf, rows.spc);
            rows.template values<kVPWin>(vf, pf, nb);
        }
    }

    // ---- merge the four waves' states through LDS -----------------------------
    constexpr int NR = 16 * RT;
    float* st = reinterpret_cast<float*>(smem);              // [4][NR][D], then [4][NR] m, l
    float* sm = st + kWaveWaves * NR * D;
    float* sl = sm + kWaveWaves * NR;
    __syncthreads();                                         // every wave is done with its meta
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float l = row4_sum(rows.l[rt]);
        const int r = wave * NR + 16 * rt + col;
#pragma unroll
        for (int nb = 0; nb < D / 16; ++nb) {
            const f32x4_t o = rows.O[rt][nb];
            *reinterpret_cast<float4*>(st + r * D + 16 * nb + 4 * gq) =
                make_float4(o[0], o[1], o[2], o[3]);
        }
        if (gq == 0) {
            sm[r] = rows.m[rt];
            sl[r] = l;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NR * (D / 4); e += kWaveBlock) {
        const int i = e / (D / 4), d = 4 * (e % (D / 4)), r = row0 + i;
        if (r >= a.rows) continue;
        float M = -FLT_MAX, L = 0.f;
#pragma unroll
        for (int w = 0; w < kWaveWaves; ++w) M = fmaxf(M, sm[w * NR + i]);
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < kWaveWaves; ++w) {
            const float f = exp2_fast(sm[w * NR + i] - M);
            const float4 o = *reinterpret_cast<const float4*>(st + (w * NR + i) * D + d);
            L = fmaf(f, sl[w * NR + i], L);
            acc.x = fmaf(f, o.x, acc.x);
            acc.y = fmaf(f, o.y, acc.y);
            acc.z = fmaf(f, o.z, acc.z);
            acc.w = fmaf(f, o.w, acc.w);
        }
        const RowDst dst = row_dst(a, b, kvh, bh, r, split, M, L, d == 0);
        dst.store4(d, acc.x, acc.y, acc.z, acc.w);
    }
    __syncthreads();                                         // (another walk may follow)
    return rows.bad;
}

template <int D, int RT, bool R16>
__global__ __launch_bounds__(kWaveBlock) __attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1)))
void attn_rows_wave_kernel(RowsLaunch a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int split = blockIdx.x % a.n_splits, rblock = blockIdx.x / a.n_splits;
    const int kvh = blockIdx.y, b = blockIdx.z;
    const int64_t bh = (int64_t)b * a.Hkv + kvh;
    const int row0 = rblock * a.block_rows;
    const Range rg(a, split, b, row0 + a.block_rows - 1);
    bool bad = false;
    // (every wave holds the same rows, so the answer is the workgroup's)
    if (!wide_queries<D, RT>(a, row0, b, kvh))
        bad = walk_wave<D, RT, 1, R16, false>(a, smem, rg, row0, bh, b, kvh, split);
    else
        bad = walk_wave<D, RT, 3, R16, false>(a, smem, rg, row0, bh, b, kvh, split);
    int* word = reinterpret_cast<int*>(smem);
    bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (threadIdx.x % kWave == 0) word[threadIdx.x / kWave] = bad;
    __syncthreads();
    bad = word[0] | word[1] | word[2] | word[3];
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(bad), 0)) {
        __syncthreads();                       // (every wave has read the words)
        for (int rt = 0; rt < RT && row0 + 16 * rt < a.rows; ++rt)
            walk_wave<D, 1, 3, R16, true>(a, smem, rg, row0 + 16 * rt, bh, b, kvh, split);
    }
}

// Merges the split partials: one wave per query row.  Each sum runs as four, of
// every fourth split: up to 64 splits of even weight, added one after the
// other, would round at the sum's full size each time.
__global__ __launch_bounds__(256) void attn_rows_merge_kernel(RowsLaunch a) {
    const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (row >= (int64_t)a.B * a.Hkv * a.rows) return;
    const int S = a.n_splits, D = a.D;
    const float* ml = a.part_ml + row * S * 2;
    float M = -FLT_MAX;
    for (int s = 0; s < S; ++s) M = fmaxf(M, ml[2 * s]);
    const int64_t bh = row / a.rows;
    const int64_t out = out_offset(a, (int)(bh / a.Hkv), (int)(bh % a.Hkv), (int)(row % a.rows));
    const float* po = a.part_o + row * S * D;
    for (int d = 4 * lane; d < D; d += 4 * kWave) {
        float4 acc[4];
        float L[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            L[i] = 0.f;
        }
        auto add = [&](int i, int s) {
            const float f = exp2_fast(ml[2 * s] - M);
            const float4 o = *reinterpret_cast<const float4*>(po + (int64_t)s * D + d);
            L[i] = fmaf(f, ml[2 * s + 1], L[i]);
            acc[i].x = fmaf(f, o.x, acc[i].x);
            acc[i].y = fmaf(f, o.y, acc[i].y);
            acc[i].z = fmaf(f, o.z, acc[i].z);
            acc[i].w = fmaf(f, o.w, acc[i].w);
        };
        int s = 0;
#pragma unroll 2
        for (; s + 4 <= S; s += 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) add(i, s + i);
        }
        for (; s < S; ++s) add(0, s);
        const float l = (L[0] + L[1]) + (L[2] + L[3]);
        const float f = l > 0.f || l != l ? 1.f / l : 0.f;      // 0: every position hidden
        auto sum = [&](float a0, float a1, float a2, float a3) { return ((a0 + a1) + (a2 + a3)) * f; };
        store4_as(a.out, out + d,
                  make_float4(sum(acc[0].x, acc[1].x, acc[2].x, acc[3].x),
                              sum(acc[0].y, acc[1].y, acc[2].y, acc[3].y),
                              sum(acc[0].z, acc[1].z, acc[2].z, acc[3].z),
                              sum(acc[0].w, acc[1].w, acc[2].w, acc[3].w)), a.io_dt);
    }
}

// Rows per kv head that the wave kernel takes: those of one workgroup, and at
// head_dim 64 of two.  us per call, wave / shared, bf16 (fp32 queries alike):
// head_dim 128 (B=8, 4K; B=1, 8K) 32 rows 48 / 58, 31 / 32, 36 rows 67 / 60, 42 /
// 32, 64 rows 68 / 63, 44 / 35; head_dim 64 (B=8, 12 heads, 2K) 40 rows 45 / 51, 64
// rows 47 / 55, 80 rows 66 / 56; head_dim 256 (B=4, 4K) 16 rows 38 / 52, 24 rows
// 63 / 55.
int few_rows(int D) { return D <= 64 ? 64 : D <= 128 ? 32 : 16; }

template <int D, bool R16>
int launch_rows(const RowsLaunch& a, hipStream_t st) {
    const dim3 grid(a.row_blocks * a.n_splits, a.Hkv, a.B);
    if (a.rows <= few_rows(D)) {
        using S = WaveShape<D>;
        if (a.block_rows == 16)
            attn_rows_wave_kernel<D, 1, R16><<<grid, kWaveBlock, S::LDS, st>>>(a);
        else
            attn_rows_wave_kernel<D, S::RT, R16><<<grid, kWaveBlock, S::LDS, st>>>(a);
    } else {
        using S = SharedShape<D>;
        if (a.block_rows == 16 * S::WAVES)
            attn_rows_shared_kernel<D, 1, R16><<<grid, S::BLOCK, S::LDS, st>>>(a);
        else
            attn_rows_shared_kernel<D, S::RT, R16><<<grid, S::BLOCK, S::LDS, st>>>(a);
    }
    int rc = check_launch("packed_attention (rows)");
    if (rc || a.n_splits == 1) return rc;
    const int64_t rows = (int64_t)a.B * a.Hkv * a.rows;
    attn_rows_merge_kernel<<<(unsigned)((rows + 3) / 4), 256, 0, st>>>(a);
    return check_launch("packed_attention (rows merge)");
}

}  // namespace

// Rows per workgroup, row blocks and splits of a call: 16 or 32 rows per
// workgroup of the wave kernel; 128 or 256 of the shared one (64 at head_dim
// 256).  Splits then give every CU a workgroup (two of the wave kernel) while
// each split keeps at least 12 units of 32 tokens.  A caller's count is followed
// while the splits' partials, which hold all rows of the call at once, fit 64 MB
// (the plan's own never take more than 34; 256 splits of 512 tokens of 32
// heads would take 2.2 GB).
RowsPlan rows_plan(int B, int Hkv, int rows, int D, int G, int n_chunks, int res_len,
                   int splits_hint) {
    constexpr int kCUs = 256, kMinUnits = 12;
    constexpr int64_t kMostPartials = 64 << 20;
    RowsPlan p;
    const bool few = rows <= few_rows(D);
    if (few) p.block_rows = rows > 16 && D <= 128 ? 32 : 16;
    else p.block_rows = D > 128 ? 64 : rows > 128 ? 256 : 128;
    p.row_blocks = (rows + p.block_rows - 1) / p.block_rows;
    const int packed = n_chunks * (G / kUnit), window = (res_len + kUnit - 1) / kUnit;
    p.n_units = packed + window;
    const int weight = packed + kWindowWeight * window;
    const int64_t groups = (int64_t)B * Hkv * p.row_blocks;
    int64_t s = splits_hint;
    if (s <= 0) s = min((few ? 2 : 1) * kCUs / groups, (int64_t)p.n_units / kMinUnits);
    s = min(s, kMostPartials / ((int64_t)B * Hkv * rows * (D + 2) * (int64_t)sizeof(float)));
    s = max((int64_t)1, min(s, (int64_t)p.n_units));
    p.weight_per_split = (int)((weight + s - 1) / s);
    p.n_splits = (weight + p.weight_per_split - 1) / p.weight_per_split;
    return p;
}

int launch_attention_rows(const RowsLaunch& a, hipStream_t st) {
    const bool r16 = a.res_dt != kSrcF32;
    switch (a.D) {
        case 64: return r16 ? launch_rows<64, true>(a, st) : launch_rows<64, false>(a, st);
        case 128: return r16 ? launch_rows<128, true>(a, st) : launch_rows<128, false>(a, st);
        case 256: return r16 ? launch_rows<256, true>(a, st) : launch_rows<256, false>(a, st);
        default: return set_error(kErrUnsupported, "head_dim %d", a.D);
    }
}

}  // namespace kivi
