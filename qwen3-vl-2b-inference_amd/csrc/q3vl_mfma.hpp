// q3vl_mfma.hpp -- device pieces the MFMA kernels share: the activation
// quantizer of one (row, group) by a quad of lanes, the widening of int8
// weights to fp16, and loads with an LDS destination.
#pragma once

#include "q3vl_device.hpp"

namespace q3vl {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define Q3VL_QUAD(v, ctrl) \
    __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true))

// The reference quantizer (cpu_f32a_i8f32sb_f32c_avx2.cpp:135-177) of one
// (row, group) by a quad of lanes: lane j holds x[16v + 4j + c] (cv[v].c), so
// chains 4j + c of the 16 run in the lane over v ascending; V[i] = P[i] +
// P[i+8] takes lane j + 2, the fixed tree runs in lane 0. The 4-value pieces
// go out as fp16 through store(v, halves), the scale from lane 0.
template <int GS, typename Store>
Q3VL_INLINE float quant_team(const float4 (&cv)[GS / 16], Store store) {
    float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;
#pragma unroll
    for (int v = 0; v < GS / 16; ++v) {
        p0 = fmaf(cv[v].x, cv[v].x, p0);
        p1 = fmaf(cv[v].y, cv[v].y, p1);
        p2 = fmaf(cv[v].z, cv[v].z, p2);
        p3 = fmaf(cv[v].w, cv[v].w, p3);
    }
    // lanes 0, 1 take lanes 2, 3 (quad_perm [2,3,2,3]); lane 0 takes lane 1's
    // V[4..7] ([1,1,1,1]); lane 0's sum to the quad ([0,0,0,0])
    const float v0 = p0 + Q3VL_QUAD(p0, 0xEE), v1 = p1 + Q3VL_QUAD(p1, 0xEE);
    const float v2 = p2 + Q3VL_QUAD(p2, 0xEE), v3 = p3 + Q3VL_QUAD(p3, 0xEE);
    const float w0 = Q3VL_QUAD(v0, 0x55), w1 = Q3VL_QUAD(v1, 0x55);
    const float w2 = Q3VL_QUAD(v2, 0x55), w3 = Q3VL_QUAD(v3, 0x55);
    const float sumsq = Q3VL_QUAD(tree8(v0, v1, v2, v3, w0, w1, w2, w3), 0x00);
    const float s = group_scale(sumsq, 1.0f / (float)GS);
    const float inv = rcp_rn(s);
    // q = rne(x / s): for a finite scale |q| < 2^11, and adding and removing
    // 1.5 * 2^23 rounds to the integer, ties to even (quant_pair_finite's
    // integer); otherwise the reference's saturating conversion
    if (__builtin_expect(__builtin_isfinite(s), 1)) {
        constexpr float kMagic = 12582912.0f;
#pragma unroll
        for (int v = 0; v < GS / 16; ++v) {
            const float r0 = (cv[v].x * inv + kMagic) - kMagic, r1 = (cv[v].y * inv + kMagic) - kMagic;
            const float r2 = (cv[v].z * inv + kMagic) - kMagic, r3 = (cv[v].w * inv + kMagic) - kMagic;
            store(v, __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r0, r1)),
                  __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r2, r3)));
        }
    } else {
#pragma unroll
        for (int v = 0; v < GS / 16; ++v) {
            const uint32_t q0 = quant_pair(cv[v].x * inv, cv[v].y * inv);
            const uint32_t q1 = quant_pair(cv[v].z * inv, cv[v].w * inv);
            store(v,
                  __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz((float)(int16_t)(q0 & 0xFFFF),
                                                                          (float)(int16_t)(q0 >> 16))),
                  __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz((float)(int16_t)(q1 & 0xFFFF),
                                                                          (float)(int16_t)(q1 >> 16))));
        }
    }
    return s;
}

// 4 int8 bytes -> 4 fp16 values in two dwords (bytes 0, 1 -> lo, 2, 3 -> hi),
// one conversion a byte: v_cvt_f16_i16 reading the byte sign-extended (SDWA
// source select) and writing one half of the destination, exact for every
// int8. The two destinations alternate, so no instruction reads the half that
// the one right before it wrote.
Q3VL_INLINE void widen4(uint32_t x, uint32_t &lo, uint32_t &hi) {
    asm("v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3"
        : "=&v"(lo), "=&v"(hi)
        : "v"(x));
}
Q3VL_INLINE half8_t widen8(uint32_t x, uint32_t y) {
    uint32_t a, b, c, d;
    widen4(x, a, b);
    widen4(y, c, d);
    return __builtin_bit_cast(half8_t, (u32x4){a, b, c, d});
}

// Loads with an LDS destination: lane l's 16 (4) bytes at voff + soff of the
// resource go to LDS at lds + 16 l (4 l). Written in asm because the compiler
// would wait for every such load before any later LDS read; dma_wait<N>()
// waits until at most N of this wave's loads are in flight (they complete in
// order).
typedef uint32_t rsrc_t __attribute__((ext_vector_type(4)));
Q3VL_INLINE rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    const uint64_t a = (uint64_t)p;
    return (rsrc_t){(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
Q3VL_INLINE void dma16(rsrc_t r, int voff, int soff, int lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
#endif
}
// (the same for bytes read once: kept out of the caches' way)
Q3VL_INLINE void dma16_nt(rsrc_t r, int voff, int soff, int lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
#endif
}
Q3VL_INLINE void dma4(rsrc_t r, int voff, int soff, int lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
#endif
}
template <int N> Q3VL_INLINE void dma_wait() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N < 63 ? N : 63) : "memory");  // (the counter's field)
#endif
}

}  // namespace q3vl
