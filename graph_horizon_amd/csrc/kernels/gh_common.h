// Device helpers shared by the gfx950 kernels.
#ifndef GH_COMMON_H
#define GH_COMMON_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gh_kargs.h"

typedef _Float16 gh_h2 __attribute__((ext_vector_type(2)));

#define GH_KERNEL extern "C" __global__

__device__ __forceinline__ float gh_h2f(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}

__device__ __forceinline__ uint16_t gh_f2h(float v) {
    // v_cvt_f16_f32 under the default round-to-nearest-even mode (f16 denormals preserved).
    // A NaN keeps its sign and the top bits of its payload, quieted — as the reference's
    // buffer writes narrow through F16C vcvtps2ph (backend/cpu/f16.rs:86-102).
    return __builtin_bit_cast(uint16_t, (_Float16)v);
}

__device__ __forceinline__ gh_h2 gh_as_h2(uint32_t v) { return __builtin_bit_cast(gh_h2, v); }

// D = a.lo*b.lo + a.hi*b.hi + c in FP32 (v_dot2_f32_f16).
__device__ __forceinline__ float gh_dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2(gh_as_h2(a), gh_as_h2(b), c, false);
}

// Workgroup barrier that orders LDS accesses only: unlike __syncthreads() (whose workgroup
// fence waits for every outstanding global load and store, vmcnt(0)), global accesses stay
// in flight across it.
__device__ __forceinline__ void gh_lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}


#define GH_GLOBAL __attribute__((address_space(1)))

// Global-address-space views of a device address (global_load/global_store, not flat).
template <class T>
__device__ __forceinline__ const GH_GLOBAL T* gh_gp(uint64_t a) {
    return (const GH_GLOBAL T*)a;
}
template <class T>
__device__ __forceinline__ GH_GLOBAL T* gh_gpw(uint64_t a) {
    return (GH_GLOBAL T*)a;
}

#define GH_DPP(v, ctrl, rmask) \
    __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rmask, 0xF, false))

// Sum across a wavefront with DPP (quad perms, half-row/row mirrors, row broadcasts); the
// total lands in lanes 48..63 (read it from lane 63).
__device__ __forceinline__ float gh_wave_sum63(float v) {
    v += GH_DPP(v, 0xB1, 0xF);   // quad_perm [1,0,3,2]
    v += GH_DPP(v, 0x4E, 0xF);   // quad_perm [2,3,0,1]
    v += GH_DPP(v, 0x141, 0xF);  // row_half_mirror
    v += GH_DPP(v, 0x140, 0xF);  // row_mirror
    v += GH_DPP(v, 0x142, 0xA);  // row_bcast:15 into rows 1 and 3
    v += GH_DPP(v, 0x143, 0xC);  // row_bcast:31 into rows 2 and 3
    return v;
}

// Maximum across a wavefront with the same DPP steps (lanes a step does not write keep their
// own value); the maximum lands in lane 63.
#define GH_DPP_KEEP(v, ctrl, rmask) \
    __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), ctrl, rmask, 0xF, false))
__device__ __forceinline__ float gh_wave_max63(float v) {
    v = fmaxf(v, GH_DPP_KEEP(v, 0xB1, 0xF));
    v = fmaxf(v, GH_DPP_KEEP(v, 0x4E, 0xF));
    v = fmaxf(v, GH_DPP_KEEP(v, 0x141, 0xF));
    v = fmaxf(v, GH_DPP_KEEP(v, 0x140, 0xF));
    v = fmaxf(v, GH_DPP_KEEP(v, 0x142, 0xA));
    v = fmaxf(v, GH_DPP_KEEP(v, 0x143, 0xC));
    return v;
}

__device__ __forceinline__ float gh_lane63(float v) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Sum / maximum across the 64 lanes of a wavefront, returned to every lane (DPP steps, then
// lane 63 read into a scalar: no LDS round trips, unlike lane shuffles through ds_bpermute).
__device__ __forceinline__ float gh_wave_sum(float v) { return gh_lane63(gh_wave_sum63(v)); }
__device__ __forceinline__ float gh_wave_max(float v) { return gh_lane63(gh_wave_max63(v)); }

// silu_mul of one FP16 gate/up pair (cpu/kernels/elementwise/activation.rs:16-29):
// f16(f16(g / (1 + e^-g)) · u) in FP32, contraction off.
__device__ __forceinline__ uint16_t gh_silu_mul_h(uint32_t g16, uint32_t u16) {
#pragma clang fp contract(off)
    const float g = gh_h2f(g16), u = gh_h2f(u16);
    const float silu = g / (1.0f + expf(-g));
    return gh_f2h(gh_h2f(gh_f2h(silu)) * u);
}

// RMSNorm scale of one FP32 row over a 256-thread workgroup, in one fixed order (each thread
// sums its float4 chunks tid, tid + 256, ... as (x²+y²)+(z²+w²); DPP wave sums; the four wave
// sums added in wave order), so every kernel that uses it gets the same bits:
// 1 / sqrt(Σx²/dim + eps) (normalization.rs:12-40). `red` is 4 floats of LDS; `s` is the
// thread's own partial. Ends with a workgroup barrier.
__device__ __forceinline__ float gh_rms_add(float s, const float4& v) {
#pragma clang fp contract(off)
    return s + ((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
}

__device__ __forceinline__ float gh_rms_finish_256(float s, uint32_t dim, float eps, float* red) {
#pragma clang fp contract(off)
    s = gh_wave_sum63(s);
    if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float sum = ((red[0] + red[1]) + red[2]) + red[3];
    return 1.0f / __builtin_sqrtf(sum / (float)dim + eps);
}

// Σx² order: thread t adds the float4 chunks of the 16-value items j = t, t + 256, ... (chunks
// 4j .. 4j + 3 in turn), then the wave sums and the four waves' sums in order — the order the
// fused RMSNorm GEMVs use, so both produce the same inverse.
__device__ __forceinline__ float gh_rms_inverse_256(const __attribute__((address_space(1))) float4* x,
                                                   uint32_t dim, float eps, float* red) {
    float s = 0.0f;
    const uint32_t n4 = dim >> 2;
    for (uint32_t j = threadIdx.x; 4 * j < n4; j += 256)
        for (uint32_t q = 0; q < 4 && 4 * j + q < n4; ++q) s = gh_rms_add(s, x[4 * j + q]);
    return gh_rms_finish_256(s, dim, eps, red);
}

// get_scale_min_k4 on the 12 scale bytes held in bytes 4..15 of the Q4_K header chunk
// (backend/cpu/dequant.rs:78-89): 6-bit (sc, mn) of sub-block j.
// Branch-free (j differs across the lanes of a wave): the scale bytes sit in hd.y (scales[0..3]),
// hd.z ([4..7]) and hd.w ([8..11]); sub-block j and j + 4 use byte j & 3 of each word, so three
// shifts by 8·(j & 3) serve both forms and a mask selects one.
__device__ __forceinline__ void gh_q4k_scale_min(const uint4& hd, uint32_t j, uint32_t& sc,
                                                 uint32_t& mn) {
    const uint32_t sh = (j & 3u) * 8u;
    const uint32_t ys = hd.y >> sh, zs = hd.z >> sh, ws = hd.w >> sh;
    const uint32_t hi = 0u - ((j >> 2) & 1u);  // all ones for j >= 4
    sc = ((ys & 63u) & ~hi) | (((ws & 15u) | ((ys >> 2) & 48u)) & hi);
    mn = ((zs & 63u) & ~hi) | ((((ws >> 4) & 15u) | ((zs >> 2) & 48u)) & hi);
}

// FP16 weights of the prefill GEMMs, a block's quants two at a time. (Whole units behind one function,
// its 16 dwords returned through references, cost the tiles 128 wait states a unit: 128 x 4096 ->
// 2 x 12288 45.0 instead of 44.4 us.)
// Q4_K: the scale and minimum of sub-blocks 2 g (low nibbles of a group) and 2 g + 1 (high ones).
// d·sc and dmin·mn are exact in FP32 (an FP16 times a 6-bit integer), and so is (d·sc)·q for a 4-bit
// q (at most 21 significant bits): the reference's product, then difference, rounds once, as one FMA
// does, so the FMA gives the same FP32 value.
struct GhW16Q4K {
    float d1, m1, d2, m2;
};
__device__ __forceinline__ GhW16Q4K gh_w16_q4k_scales(const uint4& hd, uint32_t g) {
    uint32_t sc0, mn0, sc1, mn1;
    gh_q4k_scale_min(hd, 2 * g, sc0, mn0);
    gh_q4k_scale_min(hd, 2 * g + 1, sc1, mn1);
    const float d = gh_h2f(hd.x & 0xFFFFu), dmin = gh_h2f(hd.x >> 16);
    return GhW16Q4K{d * (float)sc0, dmin * (float)mn0, d * (float)sc1, dmin * (float)mn1};
}
// Bytes e and e + 1 of q4 (a nibble each) as weights.
__device__ __forceinline__ uint32_t gh_w16_q4k_pair(uint32_t q4, int e, float sc, float mn) {
#pragma clang fp contract(off)
    typedef _Float16 hv2 __attribute__((ext_vector_type(2)));
    const float f0 = (float)((q4 >> (8 * e)) & 0xFFu), f1 = (float)((q4 >> (8 * e + 8)) & 0xFFu);
    float v0 = __builtin_fmaf(sc, f0, -mn), v1 = __builtin_fmaf(sc, f1, -mn);
    // the FP32 values are rounded to FP16 as a second step (v_cvt_pk_f16_f32), not fused
    // into one rounding of the exact value (v_fma_mix), which differs on FP16 ties
    asm volatile("" : "+v"(v0), "+v"(v1));
    const hv2 r = {(_Float16)v0, (_Float16)v1};
    return __builtin_bit_cast(uint32_t, r);
}

// Q6_K: the scales of quarters `part` (low nibbles of ql plane `part`, qh bits 2 part, 2 part + 1) and
// part + 2 (high nibbles, qh bits 4 + 2 part, 5 + 2 part) of unit (segment s, half h) and their -32-fold.
// Scale of quarter q: int8 scales[8 s + h + 2 q]; dh = the block's FP16 scale.
struct GhW16Q6K {
    float da, db, na, nb;
};
__device__ __forceinline__ GhW16Q6K gh_w16_q6k_scales(const uint4& sc, uint32_t dh, uint32_t s, uint32_t h,
                                                      uint32_t part) {
    const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
    const uint32_t ia = 8 * s + h + 2 * part, ib = ia + 4;
    const float d = gh_h2f(dh);
    const float da = d * (float)(int8_t)(scw[ia >> 2] >> (8 * (ia & 3u)));
    const float db = d * (float)(int8_t)(scw[ib >> 2] >> (8 * (ib & 3u)));
    return GhW16Q6K{da, db, -32.0f * da, -32.0f * db};
}
// Four quants of either quarter in a dword's bytes, unsigned: the nibbles with the two high bits moved
// to bits 4-5 of their byte in one shift: ((qh >> 2 part) & 3) << 4 = (qh << (4 - 2 part)) & 0x30,
// ((qh >> (4 + 2 part)) & 3) << 4 = (qh >> 2 part) & 0x30 (part is 0 or 1).
__device__ __forceinline__ uint32_t gh_w16_q6k_low(uint32_t ql, uint32_t qh, uint32_t part) {
    return (ql & 0x0F0F0F0Fu) | ((qh << (4 - 2 * part)) & 0x30303030u);
}
__device__ __forceinline__ uint32_t gh_w16_q6k_high(uint32_t ql, uint32_t qh, uint32_t part) {
    return ((ql >> 4) & 0x0F0F0F0Fu) | ((qh >> (2 * part)) & 0x30303030u);
}
// Bytes e and e + 1 of q4 as weights: (u - 32)·da = u·da + (-32·da) (the bias exact: a power-of-two
// multiple), one fused multiply-add rounded once to FP16.
__device__ __forceinline__ uint32_t gh_w16_q6k_pair(uint32_t q4, int e, float sc, float bias) {
#pragma clang fp contract(off)
    typedef _Float16 hv2 __attribute__((ext_vector_type(2)));
    const float f0 = (float)((q4 >> (8 * e)) & 0xFFu), f1 = (float)((q4 >> (8 * e + 8)) & 0xFFu);
    const hv2 r = {(_Float16)__builtin_fmaf(f0, sc, bias), (_Float16)__builtin_fmaf(f1, sc, bias)};
    return __builtin_bit_cast(uint32_t, r);
}

#endif
