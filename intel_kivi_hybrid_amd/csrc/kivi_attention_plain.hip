// Packed-KV attention over plain-layout stores (head dims or group sizes
// outside the matrix-core code order): up to 8 query rows per kv head and
// launch, in fp32.
//
// The codes are multiplied as they are, the factors folded once per chunk:
//   s[h,t] = sum_d (q ks)[h,d] c[t,d] + sum_d q[h,d] kz[d]
//   o[h,d] = sum_t (p vs)[h,t,g(d)] c'[t,d] + sum_t p[h,t] vz[t,g(d)]
// so an element costs a conversion and HG multiply-adds on each side.  A wave
// takes whole chunks, all 64 lanes busy on both sides:
// * keys [G][D/4]: 64/G lanes (4, 2 or 1) share a token's row, a code dword (16
//   channels) at a time in turn; (q ks) comes from LDS, the same float4 for
//   all tokens;
// * values [D][G/4]: a lane's items are dwords of 16 tokens of one channel,
//   consecutive in memory; (p vs) comes from LDS, the same for the channels
//   of a group.
// Each chunk's value sum starts at its correction and is formed apart before
// it is added to the output: adding c' >= 0 terms straight to the output would
// let it grow to ~1.5 sum p vs and cancel in the end (long contexts of
// near-uniform weights: 100 times the rounding).
// The next chunk's codes, scales and zeros are loaded while this one is used.
// The window is taken in passes of 16 tokens, 4 lanes per token.
//
// What bounds it: vector work (half of the ~480 instructions of a chunk at
// head_dim 96 and one row are the elements', 1 per element and side plus the
// conversion), then what a wave pays once (a third of its time at 4 chunks per
// wave).  Measured (MI355X, head_dim 96, G = 32, 4K context, B=4, 32/32 heads):
// 112 us per call with the generic kernel, which read each factor from LDS
// singly and kept half of the lanes idle, 29 us with this one (kernel 24 us,
// merge 4.7 us; 57.7 MB, 2.4 TB/s in the kernel).
#include <math.h>

#include "kivi_attention.hpp"
#include "kivi_common.hpp"
#include "kivi_mfma.hpp"

namespace kivi {
namespace {

constexpr int kPlainWaves = 4, kPlainBlock = kPlainWaves * kWave;
constexpr int kPassTokens = 16;
constexpr float kMaxMove = 8.0f;       // log2 units: the running maximum moves beyond this

// acc[h] += sum of the word's 16 codes times f[h][0..15]: byte b, bits 2k hold
// element 4b + k.
template <int HG>
__device__ __forceinline__ void mul_word(uint32_t word, const float* f, int stride, float* acc) {
    float c[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t y = (word >> (2 * k)) & 0x03030303u;
        c[k] = (float)(y & 0xffu);
        c[4 + k] = (float)((y >> 8) & 0xffu);
        c[8 + k] = (float)((y >> 16) & 0xffu);
        c[12 + k] = (float)(y >> 24);
    }
#pragma unroll
    for (int h = 0; h < HG; ++h) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float4 x = *reinterpret_cast<const float4*>(f + h * stride + 4 * b);
            acc[h] = fmaf(x.x, c[4 * b], acc[h]);
            acc[h] = fmaf(x.y, c[4 * b + 1], acc[h]);
            acc[h] = fmaf(x.z, c[4 * b + 2], acc[h]);
            acc[h] = fmaf(x.w, c[4 * b + 3], acc[h]);
        }
    }
}

// LDS of one wave (floats): q ks [HG][D], weights [HG][64], p vs
// [HG][D/Gv][G + 4], corrections [HG][D/Gv][G/16].  The wave's final state (o
// [HG][D], m, l) overlaps it.
struct PlainLds {
    int qs, p, pv, zc, floats;
    __host__ __device__ PlainLds(int HG, int D, int G, int Gv) {
        const int ng = D / Gv;
        qs = 0;
        p = HG * D;
        pv = p + HG * kWave;
        zc = pv + HG * ng * (G + 4);
        floats = (zc + HG * ng * (G / 16) + 3) / 4 * 4;
        const int state = HG * D + 2 * HG;
        if (floats < state) floats = (state + 3) / 4 * 4;
    }
};

// Waves per SIMD (and so workgroups per CU) that the registers of an instance
// allow; the split plan fills the chip with that many.
__host__ __device__ constexpr int plain_waves(int HG, int N, int J) {
    if (J == 4) return HG * N <= 4 ? 3 : HG * N <= 16 && N < 16 ? 2 : 1;
    return HG * N <= 4 ? 4 : HG * N <= 12 ? 3 : HG * N <= 32 ? 2 : 1;
}

// HG query rows; N code dwords per lane and side of a chunk; J: D and D/Gv * G
// are at most 64 J.
template <int HG, int N, int J>
__global__ __launch_bounds__(kPlainBlock)
__attribute__((amdgpu_waves_per_eu(plain_waves(HG, N, J)))) void attn_plain_kernel(AttnLaunch a) {
    extern __shared__ __align__(16) float lds[];
    const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int D = a.D, G = a.G, ng = D / a.Gv, gw = G / 16;
    const PlainLds L(HG, D, G, a.Gv);
    float* sq = lds;                                       // scaled q [HG][D]
    float* mine = lds + HG * D + wave * L.floats;
    float *qs = mine + L.qs, *sp = mine + L.p, *pv = mine + L.pv, *zc = mine + L.zc;
    const int64_t bh = (int64_t)b * a.Hkv + kvh;
    const int kv_lo = __builtin_amdgcn_readfirstlane(a.kv_start ? a.kv_start[b] : 0);
    const uint32_t* hid_row = a.hidden ? a.hidden + b * a.hidden_stride : nullptr;

    // this wave's chunks: split's range dealt in turn
    const int c_begin = split * kPlainWaves * a.chunks_per_wave;
    const int c_end = min(c_begin + kPlainWaves * a.chunks_per_wave, a.n_chunks);
    const int c_first = c_begin + wave;

    // key side: lane takes dwords part, part + lpt, ... of token kt's row
    const int lpt = G <= 16 ? 4 : G <= 32 ? 2 : 1;
    const int kt = lane / lpt, part = lane % lpt, nd = D / 16;
    const bool tok = kt < G;
    const int pv_group = (G + 4);
    uint32_t kw[N], vw[N];
    float ks[J], kz[J], vs[J], vz[J];
    const int n_items = D * gw, n_meta = ng * G;
    // this lane's bytes within a chunk (clamped to it)
    uint32_t k_off[N], v_off[N], d_off[J], e_off[J];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        k_off[i] = 4u * ((tok ? kt : 0) * nd + min(part + lpt * i, nd - 1));
        v_off[i] = 4u * min(lane + kWave * i, n_items - 1);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        d_off[j] = 4u * min(lane + kWave * j, D - 1);
        e_off[j] = 4u * min(lane + kWave * j, n_meta - 1);
    }
    auto load_keys = [&](int c) {
        const int64_t cid = bh * a.Cmax + c;
        const gptr kc = (gptr)a.k_codes + cid * (G * D / 4);
#pragma unroll
        for (int i = 0; i < N; ++i) kw[i] = gload<uint32_t>(kc, k_off[i]);
        const gptr ksp = (gptr)(a.k_scale + cid * D), kzp = (gptr)(a.k_zero + cid * D);
        const gptr vsp = (gptr)(a.v_scale + cid * n_meta), vzp = (gptr)(a.v_zero + cid * n_meta);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            ks[j] = gload<float>(ksp, d_off[j]);
            kz[j] = gload<float>(kzp, d_off[j]);
            vs[j] = gload<float>(vsp, e_off[j]);
            vz[j] = gload<float>(vzp, e_off[j]);
        }
    };
    auto load_values = [&](int c) {
        const gptr vc = (gptr)a.v_codes + (bh * a.Cmax + c) * (G * D / 4);
#pragma unroll
        for (int i = 0; i < N; ++i) vw[i] = gload<uint32_t>(vc, v_off[i]);
    };
    if (c_first < c_end) {
        load_keys(c_first);
        load_values(c_first);
    }
    const int n_real = a.qr.qlen * a.qr.hg;
    for (int e = threadIdx.x; e < HG * D; e += kPlainBlock) {
        const int h = e / D, d = e % D;
        sq[e] = h < n_real ? a.q[a.qr.row(b, kvh, h, a.Hq, D) + d] * a.qscale : 0.f;
    }
    lds_barrier();

    float m[HG], l[HG], o[N][HG];          // m: the same on every lane; l: this lane's tokens
#pragma unroll
    for (int h = 0; h < HG; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i) o[i][h] = 0.f;
    }
    float ow[HG][4];                       // the window's part: channels 4 c4 .. +3
#pragma unroll
    for (int h = 0; h < HG; ++h) ow[h][0] = ow[h][1] = ow[h][2] = ow[h][3] = 0.f;
    // A new score: moves the running maximum when it is exceeded by more than
    // kMaxMove, and returns the lane's weight (0 where the token is off or its
    // score is -inf).
    auto weigh = [&](int h, float s, bool on) {
        if (__builtin_amdgcn_ballot_w64(on && s > m[h] + kMaxMove)) {
            const float top = wave_max(on ? s : -INFINITY);
            const float f = exp2_fast(m[h] - top);
            m[h] = top;
            l[h] *= f;
#pragma unroll
            for (int i = 0; i < N; ++i) o[i][h] *= f;
#pragma unroll
            for (int i = 0; i < 4; ++i) ow[h][i] *= f;
        }
        return on && s != -INFINITY ? exp2_fast(s - m[h]) : 0.f;
    };

    // value items: dword w of channel d (items in memory order)
    int it_pv[N], it_zc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int e = min(lane + kWave * i, n_items - 1);
        const int d = e / gw, w = e % gw, g = d / a.Gv;
        it_pv[i] = g * pv_group + 16 * w;
        it_zc[i] = g * gw + w;
    }
    // p vs items: token e % G of group e / G
    int e_p[J], e_pv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int e = min(lane + kWave * j, n_meta - 1);
        e_p[j] = e % G;
        e_pv[j] = e / G * pv_group + e % G;
    }
    const int qs_h = D, pv_h = ng * pv_group, zc_h = ng * gw;

    for (int c = c_first; c < c_end; c += kPlainWaves) {
        const int next = min(c + kPlainWaves, c_end - 1);
        float bias[HG];
#pragma unroll
        for (int h = 0; h < HG; ++h) bias[h] = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int d = lane + kWave * j;
            if (d < D) {
#pragma unroll
                for (int h = 0; h < HG; ++h) {
                    const float q = sq[h * D + d];
                    qs[h * qs_h + d] = q * ks[j];
                    bias[h] = fmaf(q, kz[j], bias[h]);
                }
            }
        }
#pragma unroll
        for (int h = 0; h < HG; ++h) bias[h] = wave_sum(bias[h]);
        wave_sync();
        float s[HG];
#pragma unroll
        for (int h = 0; h < HG; ++h) s[h] = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int dw = part + lpt * i;
            // (as a branch: multiplying codes of 0 instead let the compiler hold
            // every word's factors at once, and spill)
            if (dw < nd) mul_word<HG>(kw[i], qs + 16 * dw, qs_h, s);
        }
        const int pos = c * G + kt;
        const bool on = tok && pos >= kv_lo && !(hid_row && position_hidden(hid_row, pos));
#pragma unroll
        for (int h = 0; h < HG; ++h) {
            if (lpt > 1) s[h] += dpp<0xB1>(s[h]);           // quad_perm [1,0,3,2]
            if (lpt > 2) s[h] += dpp<0x4E>(s[h]);           // quad_perm [2,3,0,1]
            const float w = weigh(h, s[h] + bias[h], on);
            if (part == 0) {
                l[h] += w;
                if (tok) sp[h * kWave + kt] = w;
            }
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int e = lane + kWave * j;
            const bool in = e < n_meta;
#pragma unroll
            for (int h = 0; h < HG; ++h) {
                const float p = in ? sp[h * kWave + e_p[j]] : 0.f;
                // 16 lanes hold the 16 tokens of one dword of the group
                const float z = row_sum16(in ? p * vz[j] : 0.f);
                if (in) {
                    pv[h * pv_h + e_pv[j]] = p * vs[j];
                    if (lane % 16 == 0) zc[h * zc_h + e / 16] = z;
                }
            }
        }
        load_keys(next);
        wave_sync();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float acc[HG];
#pragma unroll
            for (int h = 0; h < HG; ++h) acc[h] = zc[h * zc_h + it_zc[i]];
            mul_word<HG>(vw[i], pv + it_pv[i], pv_h, acc);
#pragma unroll
            for (int h = 0; h < HG; ++h) o[i][h] += acc[h];
        }
        load_values(next);
    }

    // ---- the window, in passes of 16 tokens dealt over all waves, last first --
    const int f4 = D / 4, ts_n = kWave / f4, c4 = lane % f4, ts = lane / f4;
    const int n_waves = a.n_qsplits * kPlainWaves, w_idx = n_waves - 1 - (split * kPlainWaves + wave);
    const int n_pass = (a.res_len + kPassTokens - 1) / kPassTokens;
    auto window = [&](auto wide) {
        for (int pass = w_idx; pass < n_pass; pass += n_waves) {
            const int t0 = pass * kPassTokens, n = min(kPassTokens, a.res_len - t0);
            auto row = [&](int t) {
                int s = a.res_start + t0 + min(t, n - 1);
                s = s >= a.Rcap ? s - a.Rcap : s;
                return (bh * a.Rcap + s) * D;
            };
            const int tk = lane / 4, qq = lane % 4;
            const int64_t kr = row(tk) + 4 * qq;
            float s[HG];
#pragma unroll
            for (int h = 0; h < HG; ++h) s[h] = 0.f;
            float4 kv[4 * J];
#pragma unroll
            for (int j = 0; j < 4 * J; ++j) kv[j] = wide(a.k_res, kr + 16 * min(j, nd - 1));
#pragma unroll
            for (int j = 0; j < 4 * J; ++j) {
                if (j < nd) {
#pragma unroll
                    for (int h = 0; h < HG; ++h) {
                        const float4 q = *reinterpret_cast<const float4*>(sq + h * D + 4 * qq + 16 * j);
                        s[h] = fmaf(q.x, kv[j].x, s[h]);
                        s[h] = fmaf(q.y, kv[j].y, s[h]);
                        s[h] = fmaf(q.z, kv[j].z, s[h]);
                        s[h] = fmaf(q.w, kv[j].w, s[h]);
                    }
                }
            }
            const int pos = a.n_chunks * G + t0 + tk;
            const bool seen = tk < n && pos >= kv_lo && !(hid_row && position_hidden(hid_row, pos));
            wave_sync();                  // the previous pass's weights have been read
#pragma unroll
            for (int h = 0; h < HG; ++h) {
                s[h] += dpp<0xB1>(s[h]);
                s[h] += dpp<0x4E>(s[h]);
                const float w = weigh(h, s[h], seen && t0 + tk < a.qr.visible(h, a.res_len));
                if (qq == 0) {
                    l[h] += w;
                    sp[h * kWave + tk] = w;
                }
            }
            wave_sync();
            if (ts < ts_n) {
                for (int t = ts; t < n; t += ts_n) {
                    const float4 v = wide(a.v_res, row(t) + 4 * c4);
#pragma unroll
                    for (int h = 0; h < HG; ++h) {
                        const float p = sp[h * kWave + t];
                        ow[h][0] = fmaf(p, v.x, ow[h][0]);
                        ow[h][1] = fmaf(p, v.y, ow[h][1]);
                        ow[h][2] = fmaf(p, v.z, ow[h][2]);
                        ow[h][3] = fmaf(p, v.w, ow[h][3]);
                    }
                }
            }
        }
    };
    if (a.res_dt == kSrcF32) {
        window([](const void* p, int64_t i) { return load4_vec<kSrcF32>(p, i); });
    } else {
        const uint32_t half_mask = a.res_dt == kSrcF16 ? ~0u : 0u;
        window([half_mask](const void* p, int64_t i) { return load4_16(p, i, half_mask); });
    }

    // ---- the wave's state in its LDS region: o [HG][D], m [HG], l [HG] ---------
    wave_sync();
    for (int e = lane; e < HG * D; e += kWave) mine[e] = 0.f;
    wave_sync();
    for (int w = 0; w < gw; ++w) {         // a channel's dwords lie in different lanes
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int e = lane + kWave * i;
            if (e < n_items && e % gw == w) {
#pragma unroll
                for (int h = 0; h < HG; ++h) mine[h * D + e / gw] += o[i][h];
            }
        }
        wave_sync();
    }
    for (int s = 0; s < ts_n; ++s) {
        if (ts == s) {
#pragma unroll
            for (int h = 0; h < HG; ++h) {
#pragma unroll
                for (int i = 0; i < 4; ++i) mine[h * D + 4 * c4 + i] += ow[h][i];
            }
        }
        wave_sync();
    }
#pragma unroll
    for (int h = 0; h < HG; ++h) {
        const float sum = wave_sum(l[h]);
        if (lane == 0) {
            mine[HG * D + h] = m[h];
            mine[HG * D + HG + h] = sum;
        }
    }
    __syncthreads();
    const int64_t prow0 = ((int64_t)b * a.Hkv + kvh) * HG;      // partial rows
    for (int e = threadIdx.x; e < HG * D; e += kPlainBlock) {
        const int h = e / D, d = e % D;
        if (!a.qr.real(h)) continue;
        float M = -INFINITY, acc = 0.f, sum = 0.f;
        for (int w = 0; w < kPlainWaves; ++w)
            M = fmaxf(M, lds[HG * D + w * L.floats + HG * D + h]);
        for (int w = 0; w < kPlainWaves; ++w) {
            const float* st = lds + HG * D + w * L.floats;
            const float f = st[HG * D + h] == -INFINITY ? 0.f : exp2_fast(st[HG * D + h] - M);
            acc = fmaf(f, st[h * D + d], acc);
            sum = fmaf(f, st[HG * D + HG + h], sum);
        }
        if (a.n_splits == 1) {             // (a row with no visible position gives 0)
            a.out[a.qr.row(b, kvh, h, a.Hq, D) + d] = sum > 0.f ? acc / sum : 0.f;
        } else {
            const int64_t row = (prow0 + h) * a.n_splits + split;
            a.part_o[row * D + d] = acc;
            if (d == 0) {
                a.part_ml[row * 2] = M;
                a.part_ml[row * 2 + 1] = sum;
            }
        }
    }
}

template <int N, int J>
int launch_rows_of(const AttnLaunch& a, hipStream_t st) {
    const dim3 grid(a.n_splits, a.Hkv, a.B);
    const int HG = a.qr.rows;
    const size_t bytes =
        (HG * a.D + kPlainWaves * PlainLds(HG, a.D, a.G, a.Gv).floats) * sizeof(float);
    switch (HG) {
        case 1: attn_plain_kernel<1, N, J><<<grid, kPlainBlock, bytes, st>>>(a); break;
        case 2: attn_plain_kernel<2, N, J><<<grid, kPlainBlock, bytes, st>>>(a); break;
        case 4: attn_plain_kernel<4, N, J><<<grid, kPlainBlock, bytes, st>>>(a); break;
        default: attn_plain_kernel<8, N, J><<<grid, kPlainBlock, bytes, st>>>(a); break;
    }
    return check_launch("packed_attention (plain)");
}

}  // namespace

bool plain_attention_supported(int D, int G, int Gv) {
    return D % 16 == 0 && D <= 256 && G % 16 == 0 && G <= kWave && D / Gv * G <= 4 * kWave;
}

// With 1 or 2 rows, or chunks of up to 32 tokens, this kernel is ahead (the
// generic one leaves half of its lanes idle at 32 tokens and reads every factor by
// itself).  With 4 and more rows and chunks of 48 or 64 tokens, where a lane has a
// whole token, the sums of all rows for its code words and the factors leave one
// or two waves per SIMD; from 1 to 3 chunks per wave (4 rows of more than 128
// factors), from 32 chunks in all (8 rows of 48 tokens) and up to 6 per wave (8
// rows of 64) the generic kernel's many small workgroups win.  us per call, generic / this one (head_dim, G, Gv; B and
// tokens at 8 kv heads): 4 rows 42.2 / 35.8 (96, 64, 96; 4, 4K), 21.2 / 24.3 (48,
// 64, 16; 4, 4K), 35.2 / 40.7 (80, 48, 16; 4, 4K), 42.0 / 35.2 (64, 64, 16; 1, 30K); 8
// rows 50.4 / 61 (96, 64, 32; 4, 4K), 85 / 96 (1, 30K), 257 / 165 (16, 4K), 110 / 118
// (48, 48, 16; 16, 4K), 46 / 40 (96, 64, 32; 1, 200).
bool plain_attention_takes(int rows, int D, int G, int Gv, int pairs, int n_chunks) {
    if (!plain_attention_supported(D, G, Gv)) return false;
    if (G <= 32 || rows <= 2) return true;
    const int64_t chunks = (int64_t)pairs * n_chunks, per_wave = kPlainWaves * 256;
    if (rows == 4)
        return D / Gv * G <= 2 * kWave || chunks < per_wave || chunks >= 3 * per_wave;
    return chunks <= 32 || (G > 48 && chunks >= 6 * per_wave);
}

// The instance (N, J) of a geometry.
static void plain_instance(int D, int G, int Gv, int& N, int& J) {
    const int lpt = G <= 16 ? 4 : G <= 32 ? 2 : 1;
    const int n = (D / 16 + lpt - 1) / lpt;                // code dwords per lane and side
    const int meta = D > D / Gv * G ? D : D / Gv * G;
    J = meta <= kWave ? 1 : meta <= 2 * kWave ? 2 : 4;
    if (J == 1) N = n <= 2 ? 2 : 4;
    else if (J == 2) N = n <= 2 ? 2 : n <= 3 ? 3 : n <= 4 ? 4 : 8;
    else N = n <= 4 ? 4 : n <= 8 ? 8 : 16;
}

int plain_attention_groups_per_cu(int rows, int D, int G, int Gv) {
    int N, J;
    plain_instance(D, G, Gv, N, J);
    const int lds = (rows * D + kPlainWaves * PlainLds(rows, D, G, Gv).floats) * (int)sizeof(float);
    const int fit = 160 * 1024 / lds, waves = plain_waves(rows, N, J);
    return fit < waves ? (fit < 1 ? 1 : fit) : waves;
}

int launch_attention_plain(const AttnLaunch& a, hipStream_t st) {
    int N, J;
    plain_instance(a.D, a.G, a.Gv, N, J);
    if (J == 1) return N == 2 ? launch_rows_of<2, 1>(a, st) : launch_rows_of<4, 1>(a, st);
    if (J == 2) {
        if (N == 2) return launch_rows_of<2, 2>(a, st);
        if (N == 3) return launch_rows_of<3, 2>(a, st);
        return N == 4 ? launch_rows_of<4, 2>(a, st) : launch_rows_of<8, 2>(a, st);
    }
    if (N == 4) return launch_rows_of<4, 4>(a, st);
    return N == 8 ? launch_rows_of<8, 4>(a, st) : launch_rows_of<16, 4>(a, st);
}

}  // namespace kivi
