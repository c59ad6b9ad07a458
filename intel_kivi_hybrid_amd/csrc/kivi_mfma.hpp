// Building blocks shared by the packed-attention kernels: operand types, the
// bf16 MFMA, the exact splits of fp32 factors into bf16 pieces, a wave's LDS
// order and reductions across its lanes.
#pragma once

#include "kivi_common.hpp"

namespace kivi {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    bf16x2_t v = {(__bf16)a, (__bf16)b};   // round to nearest even
    return __builtin_bit_cast(uint32_t, v);
}

// The bf16 pairs (-1, 0) and (0, -1), held in VGPRs: split_pair's v_dot2
// reads them as register operands.  (As literals, the compiler's encoding of
// the (-1, 0) pair made the instruction read the pair's high half -- measured
// on gfx950 -- so the values are hidden from it.)
struct SplitConsts {
    uint32_t neg_x, neg_y;
};
__device__ __forceinline__ SplitConsts split_consts() {
    SplitConsts c{0x0000bf80u, 0xbf800000u};
    asm("" : "+v"(c.neg_x));
    asm("" : "+v"(c.neg_y));
    return c;
}

// (a, b) -> hi and lo bf16 pairs with a ~ hi.x + lo.x, b ~ hi.y + lo.y.
// a - hi.x is exact in fp32 (hi.x is a rounded to 8 significant bits), so
// one v_dot2_f32_bf16 of hi with (-1, 0) accumulated onto a forms it: two
// ops instead of widening hi's halves and subtracting (bit-identical over
// 8.4 M random pairs on gfx950, tiny normals included).
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& lo,
                                           SplitConsts k) {
    hi = pack_bf16x2(a, b);
    const bf16x2_t h2 = __builtin_bit_cast(bf16x2_t, hi);
    const float la = __builtin_amdgcn_fdot2_f32_bf16(h2, __builtin_bit_cast(bf16x2_t, k.neg_x), a,
                                                     false);
    const float lb = __builtin_amdgcn_fdot2_f32_bf16(h2, __builtin_bit_cast(bf16x2_t, k.neg_y), b,
                                                     false);
    lo = pack_bf16x2(la, lb);
}

// Three pieces: a ~ hi.x + mid.x + lo.x, b likewise (~2^-25 relative).  Each
// residual is exact in fp32 (the piece taken off is the value rounded to 8
// significant bits), so only lo's rounding remains.
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t& hi, uint32_t& mid,
                                            uint32_t& lo, SplitConsts k) {
    hi = pack_bf16x2(a, b);
    const bf16x2_t h2 = __builtin_bit_cast(bf16x2_t, hi);
    const float ra = __builtin_amdgcn_fdot2_f32_bf16(h2, __builtin_bit_cast(bf16x2_t, k.neg_x), a,
                                                     false);
    const float rb = __builtin_amdgcn_fdot2_f32_bf16(h2, __builtin_bit_cast(bf16x2_t, k.neg_y), b,
                                                     false);
    mid = pack_bf16x2(ra, rb);
    const bf16x2_t m2 = __builtin_bit_cast(bf16x2_t, mid);
    const float sa = __builtin_amdgcn_fdot2_f32_bf16(m2, __builtin_bit_cast(bf16x2_t, k.neg_x), ra,
                                                     false);
    const float sb = __builtin_amdgcn_fdot2_f32_bf16(m2, __builtin_bit_cast(bf16x2_t, k.neg_y), rb,
                                                     false);
    lo = pack_bf16x2(sa, sb);
}

// Orders a wave's LDS writes before its own later LDS reads (other lanes of
// the same wave read what a lane wrote).  A wave's LDS operations execute in
// program order, so no wait is needed for that: the fences are at wavefront
// scope, which keeps the compiler from moving LDS accesses across this point
// and emits no s_waitcnt.  (Workgroup scope made every such point wait for
// the wave's LDS writes to complete: 1.3 % slower at config 4.)  Never used
// for data passed between waves; that takes lds_barrier().
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
        0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Reductions across the 16 lanes of a DPP row (row_ror 8, 4, 2, 1).
__device__ __forceinline__ float row_max16(float v) {
    v = fmaxf(v, dpp<0x128>(v));
    v = fmaxf(v, dpp<0x124>(v));
    v = fmaxf(v, dpp<0x122>(v));
    return fmaxf(v, dpp<0x121>(v));
}

__device__ __forceinline__ float row_sum16(float v) {
    v += dpp<0x128>(v);
    v += dpp<0x124>(v);
    v += dpp<0x122>(v);
    return v + dpp<0x121>(v);
}

// Across the wave: DPP within each 16-lane row, then the four row results
// through readlane.  (__shfl_xor compiles to ds_bpermute, a chain of six LDS
// round trips.)
__device__ __forceinline__ float lane_f(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float wave_max(float v) {
    v = row_max16(v);
    return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}
__device__ __forceinline__ float wave_sum(float v) {
    v = row_sum16(v);
    return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}

}  // namespace
}  // namespace kivi
