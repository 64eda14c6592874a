// device.hpp -- device helpers shared by the kernel files: the canonical exp, cross-lane
// reductions, the 32-element int8 quantisation and the top-2 (argmax, margin) merge.
// The reduction orders they implement are listed at the top of kernels.hip.
#pragma once
#include "common.hpp"

#include <climits>

namespace mi {

// ------------------------------------------------------------------ scalar helpers
__device__ __forceinline__ float mi_expf(float x) {
    if (x != x) return x;
    if (x > 88.72283f) return __builtin_inff();
    if (x < -87.0f) return 0.0f;
    const float n = __builtin_rintf(__fmul_rn(x, 0x1.715476p+0f));
    float r = __fmaf_rn(n, -0x1.62e4p-1f, x);
    r = __fmaf_rn(n, -0x1.7f7d1cp-20f, r);
    float p = 0x1.a01a02p-13f;
    p = __fmaf_rn(p, r, 0x1.6c16c2p-10f);
    p = __fmaf_rn(p, r, 0x1.111112p-7f);
    p = __fmaf_rn(p, r, 0x1.555556p-5f);
    p = __fmaf_rn(p, r, 0x1.555556p-3f);
    p = __fmaf_rn(p, r, 0x1p-1f);
    p = __fmaf_rn(p, r, 1.0f);
    p = __fmaf_rn(p, r, 1.0f);
    return __builtin_ldexpf(p, (int)n);
}

// LDS hand-off between lanes of one wave (waves run independently, so a workgroup
// barrier cannot be used): DS operations of one wave complete in order
// (the s_waitcnt builtin, unlike inline asm, is seen by the compiler's own wait
// insertion, which then knows nothing is outstanding afterwards; gfx9 encoding:
// vmcnt in bits 3:0 + 15:14, expcnt 6:4, lgkmcnt 11:8)
__device__ __forceinline__ void wave_lds_sync() { __builtin_amdgcn_s_waitcnt(0xC07F); }   // lgkmcnt(0)
__device__ __forceinline__ float h2f_lo(uint32_t u) { return __half2float(__ushort_as_half((unsigned short)(u & 0xFFFFu))); }
__device__ __forceinline__ float h2f_hi(uint32_t u) { return __half2float(__ushort_as_half((unsigned short)(u >> 16))); }
__device__ __forceinline__ float fp16_round(float v) { return __half2float(__float2half(v)); }

// Cross-lane partners without the LDS pipe. The xor butterfly pairs lane l with
// l ^ off for off = 32, 16, ..., 1; every step leaves a pair holding the same value
// (IEEE add and max are commutative), which the cheaper permutations rely on:
//   off 32, 16: v_permlane32_swap / v_permlane16_swap of v with itself leave the two
//               values of each pair (l, l ^ off) in the two results on lane l;
//   off 8:      DPP row_ror:8 is l ^ 8 inside each 16-lane row;
//   off 4:      DPP row_ror:4 reads lane (l + 4) mod 16, which holds the value of
//               l ^ 4 once the values are symmetric under xor 8;
//   off 2, 1:   DPP quad_perm [2,3,0,1] and [1,0,3,2] are l ^ 2 and l ^ 1.
// So each step adds exactly the same two values as the xor butterfly.
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ int dppi(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppRor4 = 0x124, kDppRor8 = 0x128, kDppHalfMirror = 0x141;
__device__ __forceinline__ void pair32(float v, float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void pair16(float v, float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ float bfly_sum64(float v) {
    float a, b;
    pair32(v, a, b);
    v = __fadd_rn(a, b);
    pair16(v, a, b);
    v = __fadd_rn(a, b);
    v = __fadd_rn(v, dppf<kDppRor8>(v));
    v = __fadd_rn(v, dppf<kDppRor4>(v));
    v = __fadd_rn(v, dppf<kDppXor2>(v));
    return __fadd_rn(v, dppf<kDppXor1>(v));
}
__device__ __forceinline__ float wave_max(float v) {
    float a, b;
    pair32(v, a, b);
    v = fmaxf(a, b);
    pair16(v, a, b);
    v = fmaxf(a, b);
    v = fmaxf(v, dppf<kDppRor8>(v));
    v = fmaxf(v, dppf<kDppRor4>(v));
    v = fmaxf(v, dppf<kDppXor2>(v));
    return fmaxf(v, dppf<kDppXor1>(v));
}
// max / integer sum over aligned groups of 8 lanes (exact in any order): quad steps,
// then the half-row mirror pairs lane i of a quad with the other quad of its 8
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, dppf<kDppXor1>(v));
    v = fmaxf(v, dppf<kDppXor2>(v));
    return fmaxf(v, dppf<kDppHalfMirror>(v));
}
__device__ __forceinline__ int sum8(int v) {
    v += dppi<kDppXor1>(v);
    v += dppi<kDppXor2>(v);
    return v + dppi<kDppHalfMirror>(v);
}

// max / integer sum over each 32-lane half (exact in any order; pairings as in
// bfly_sum64: permlane16 swap, then DPP inside 16-lane rows)
__device__ __forceinline__ float max32(float v) {
    float a, b;
    pair16(v, a, b);
    v = fmaxf(a, b);
    v = fmaxf(v, dppf<kDppRor8>(v));
    v = fmaxf(v, dppf<kDppRor4>(v));
    v = fmaxf(v, dppf<kDppXor2>(v));
    return fmaxf(v, dppf<kDppXor1>(v));
}
__device__ __forceinline__ int sum32(int v) {
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    v = (int)(r[0] + r[1]);
    v += dppi<kDppRor8>(v);
    v += dppi<kDppRor4>(v);
    v += dppi<kDppXor2>(v);
    return v + dppi<kDppXor1>(v);
}

// quantize one 32-element block per half-wave: the lane's code, the block scale and
// 8*sum(q) on every lane (cuda_infer.cu:80-89, mega.cu:303-325)
__device__ __forceinline__ void quant32_vals(float v, int& q, float& d, int& s8) {
    const float a = max32(fabsf(v));
    const float inv = a > 0.f ? __fdiv_rn(127.f, a) : 0.f;
    q = __float2int_rn(__fmul_rn(v, inv));
    d = fp16_round(__fdiv_rn(a, 127.f));
    s8 = 8 * sum32(q);
}

// ------------------------------------------------------------------ argmax candidates
struct Top2 { float best; int idx; float second; };
__device__ __forceinline__ void top2_push(Top2& t, float v, int row) {   // rows arrive increasing
    if (v > t.best) { t.second = t.best; t.best = v; t.idx = row; }
    else if (v > t.second) t.second = v;
}
__device__ __forceinline__ void top2_merge(Top2& a, float ob, int oi, float os) {
    const bool take = ob > a.best || (ob == a.best && oi < a.idx);
    a.second = fmaxf(fmaxf(a.second, os), take ? a.best : ob);
    if (take) { a.best = ob; a.idx = oi; }
}
// the xor butterfly over 64 lanes with the pairings of bfly_sum64; the pair merge is
// symmetric (max, lowest index on ties), so each step gives the xor result
__device__ __forceinline__ void top2_wave(Top2& t) {
    auto swap_merge = [&](bool p32) {
        const unsigned b = __float_as_uint(t.best), i = (unsigned)t.idx, s2 = __float_as_uint(t.second);
        const auto rb = p32 ? __builtin_amdgcn_permlane32_swap(b, b, false, false) : __builtin_amdgcn_permlane16_swap(b, b, false, false);
        const auto ri = p32 ? __builtin_amdgcn_permlane32_swap(i, i, false, false) : __builtin_amdgcn_permlane16_swap(i, i, false, false);
        const auto rs = p32 ? __builtin_amdgcn_permlane32_swap(s2, s2, false, false) : __builtin_amdgcn_permlane16_swap(s2, s2, false, false);
        Top2 x{__uint_as_float(rb[0]), (int)ri[0], __uint_as_float(rs[0])};
        top2_merge(x, __uint_as_float(rb[1]), (int)ri[1], __uint_as_float(rs[1]));
        t = x;
    };
    swap_merge(true);
    swap_merge(false);
    top2_merge(t, dppf<kDppRor8>(t.best), dppi<kDppRor8>(t.idx), dppf<kDppRor8>(t.second));
    top2_merge(t, dppf<kDppRor4>(t.best), dppi<kDppRor4>(t.idx), dppf<kDppRor4>(t.second));
    top2_merge(t, dppf<kDppXor2>(t.best), dppi<kDppXor2>(t.idx), dppf<kDppXor2>(t.second));
    top2_merge(t, dppf<kDppXor1>(t.best), dppi<kDppXor1>(t.idx), dppf<kDppXor1>(t.second));
}

// The token of a merged top-2. Only when no logit compares greater than -inf (all NaN
// or -inf) is no row taken and idx left at INT_MAX; the first-max argmax of
// cpu_infer.cpp:153-154 returns row 0 then, and so does this. (It also keeps the next
// step's embedding gather, which reads row tokbuf[pos + 1], inside the table.)
__device__ __forceinline__ int top2_token(const Top2& a, int V) { return (unsigned)a.idx < (unsigned)V ? a.idx : 0; }

}  // namespace mi
