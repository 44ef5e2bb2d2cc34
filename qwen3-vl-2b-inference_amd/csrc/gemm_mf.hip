// gemm_mf.hip -- 16 or fewer activation rows against a very wide weight (the
// lm_head over a batch of rows) on 16x16 MFMA tiles, at group size 64 (gfx950).
#include "q3vl_device.hpp"
#include "q3vl_kernels.hpp"

namespace q3vl {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 4 int8 bytes -> 4 fp16 values in two dwords (bytes 0, 1 -> lo, 2, 3 -> hi),
// one conversion per byte: v_cvt_f16_i16 reading the byte sign-extended
// (SDWA source select) and writing one half of the destination (the other
// half kept), exact for every int8.
__device__ __forceinline__ void widen4_mf(uint32_t x, uint32_t &lo, uint32_t &hi) {
    asm("v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3"
        : "=&v"(lo), "=&v"(hi)
        : "v"(x));
}

// ------------------------------------------------ wide products, few rows
// 16 or fewer activation rows against a very wide weight (the lm_head over a
// batch of rows): the product is 16 rows x N, so the 32-row tiles above would
// pad it, and they stage every weight row through LDS. Here one wave computes
// 16 weight rows x the 16 activation rows with v_mfma_f32_16x16x32_f16, the
// weights going straight from the load into the MFMA operand:
// * B (weights): lane l takes weight row n = l % 16 of the tile and, of each
//   group's 64 bytes, bytes 16c .. 16c + 15 (c = l / 16) -- one 16-byte load a
//   lane and group; widened to fp16 (widen4_mf), its first 8 k feed the
//   group's first MFMA, the other 8 the second.
// * A: MFMA u of lane l takes row l % 16, k = 16c + 8u + j (j = 0..7) -- the k
//   the weight bytes hold. Each block quantizes the activations itself into
//   LDS in that lane order, 16-byte pieces [group][u][lane], and the a_s as
//   [group][row] (rows M..15 zero), so no quantizer launch precedes it: a
//   team of 4 lanes per (row, group) runs the reference quantizer
//   (i8:135-177) in its own order -- the 16 FMA chains over x[16t + i]^2,
//   P0[i] + P1[i], the fixed tree, s = sqrt(sumsq/64 + 1e-6) / 127 by
//   group_scale, q = rne(x * (1/s)) saturated to
//   int16, as fp16 (exact: |q| <= 1016 wherever s is finite).
// * G of a group is the MFMA pair's exact integer sum (every partial sum is
//   below 2^24);
//   lane l holds rows 4c + i, column n, and folds out = fma(G * a_s, w_s, out)
//   group by group in ascending order (i8:613-617, 652).
// * Each wave takes a contiguous run of 16-row tiles (the runs differ by at
//   most one tile); its loads run D quads (4 groups each) ahead, across its
//   tiles. Per tile it keeps the greedy-argmax candidate of each row
//   (am_combine over its columns; values not above -FLT_MAX never win), and
//   at the end leaves one partial per row (an empty one without tiles).
template <int D, int NW, int MINB>
__global__ __launch_bounds__(64 * NW, MINB) void gemm_mf_wide_kernel(const float *A,
                                                                 const int8_t *W, const float *S, int N,
                                                                 int K, int M, int nwaves, int ntiles,
                                                                 float *C, float *part_val,
                                                                 int32_t *part_idx) {
    constexpr int NT = 64 * NW;  // threads
    extern __shared__ __align__(16) unsigned char smem[];
    const int Kg = K / 64, qpt = Kg / 4;  // groups; quads per tile
    u32x4 *Al = reinterpret_cast<u32x4 *>(smem);                  // [Kg][2][64]
    float *asl = reinterpret_cast<float *>(smem + Kg * 2 * 64 * 16);  // [Kg][16]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gw = (int)blockIdx.x * NW + wid;  // this wave's partial
    // tiles [t0, t1): the waves' shares differ by at most one tile
    const int t0 = (int)((long)gw * ntiles / nwaves), t1 = (int)((long)(gw + 1) * ntiles / nwaves);

    constexpr int kRsrcWord3 = 0x00020000;
    const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void *)W, 0, N * K, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc((void *)S, 0, N * Kg * 4, kRsrcWord3);
    const int c = lane >> 4, nl = lane & 15;
    // weight row of tile t (clamped into the weight; columns past N are not
    // kept) and its byte offset of quad q
    u32x4 wr[D][4];
    float4 wsr[D];
    const int nq = max(t1 - t0, 0) * qpt;  // quads over the wave's tiles
    auto load = [&](int sl, int Q) __attribute__((always_inline)) {
        const int t = t0 + Q / qpt, g0 = 4 * (Q % qpt);
        const int row = min(16 * t + nl, N - 1);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            wr[sl][u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                      rW, row * K + 16 * c, 64 * (g0 + u), 0));
        wsr[sl] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rS, row * Kg * 4, 4 * g0, 0));
    };
    // ---- quantize A into LDS (every thread of the block, before its
    // barrier). A team of 4 lanes per (row, group), rows 0..RW-1, groups
    // fastest (a wave's loads read 16 consecutive 256-byte groups, 64 bytes
    // a team each); rows past M are zeros, and with RW = 8 rows 8..15 are
    // zero-filled. Lane j of a team holds x[16v + 4j + c] (v, c = 0..3):
    // the whole chains i = 4j + c of the sum of squares, t = v ascending.
    // v_i = P_i + P_{i+8} pairs lanes j and j + 2, the tree's v_i + v_{i+4}
    // lanes 0 and 1, then (s0 + s1) + (s2 + s3) in lane 0. The teams go in
    // batches of QB passes whose loads are all issued before any of them is
    // used (rows clamped into A, no branch around a load); the first batch
    // goes out ahead of the weight stream, so waiting for it leaves the
    // weights in flight.
    const int RW = M <= 8 ? 8 : 16;
    const int nteam = RW * Kg;  // a multiple of NT / 4 (Kg is a multiple of 8)
    const int tj = tid & 3;
    constexpr int QB = 4;
    float4 xb[QB][4];
    auto load_batch = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < QB; ++it) {
            const int tm = min((tid >> 2) + tb + (NT / 4) * it, nteam - 1);
            const float *xr = A + (size_t)min(tm / Kg, M - 1) * K + 64 * (tm % Kg) + 4 * tj;
#pragma unroll
            for (int v = 0; v < 4; ++v) xb[it][v] = *reinterpret_cast<const float4 *>(xr + 16 * v);
        }
    };
    load_batch(0);
    // the weight stream starts before the activations are quantized; the
    // slots are issued in ring order, as the loop reissues them (the wait
    // counts at the loop head cover both paths: any other order here would
    // make every quad's first use wait for nearly every load in flight)
    if (nq > 0) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            load(j, min(j, nq - 1));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (RW == 8) {
        for (int q = tid; q < Kg * 16; q += NT) {  // (group, u, c) pieces of rows 8..15
            const int g = q >> 4, u = (q >> 3) & 1, cc = (q >> 1) & 3, r = 8 + 4 * (q & 1);
            u32x4 *d = Al + (g * 2 + u) * 64 + 16 * cc + r;
#pragma unroll
            for (int z = 0; z < 4; ++z) d[z] = (u32x4){0u, 0u, 0u, 0u};
        }
        for (int q = tid; q < Kg * 8; q += NT) asl[(q >> 3) * 16 + 8 + (q & 7)] = 0.0f;
    }
    // batch tb's teams (their loads in xb)
    auto quant_batch = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < QB; ++it) {
            const int tm = (tid >> 2) + tb + (NT / 4) * it;
            if (tm >= nteam) break;  // wave-uniform (16 teams a wave)
            const int g = tm % Kg, m = tm / Kg;
            const bool real = m < M;
            float4 xv[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float4 f = xb[it][v];
                xv[v] = real ? f : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            float P[4];
            P[0] = fmaf(xv[0].x, xv[0].x, 0.0f);
            P[1] = fmaf(xv[0].y, xv[0].y, 0.0f);
            P[2] = fmaf(xv[0].z, xv[0].z, 0.0f);
            P[3] = fmaf(xv[0].w, xv[0].w, 0.0f);
#pragma unroll
            for (int v = 1; v < 4; ++v) {
                P[0] = fmaf(xv[v].x, xv[v].x, P[0]);
                P[1] = fmaf(xv[v].y, xv[v].y, P[1]);
                P[2] = fmaf(xv[v].z, xv[v].z, P[2]);
                P[3] = fmaf(xv[v].w, xv[v].w, P[3]);
            }
            float V[4], T[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) V[c] = P[c] + __shfl_xor(P[c], 2, 4);  // lanes 0, 1: v_{4j+c}
#pragma unroll
            for (int c = 0; c < 4; ++c) T[c] = V[c] + __shfl_xor(V[c], 1, 4);  // lane 0: s_c
            const float sumsq = __shfl((T[0] + T[1]) + (T[2] + T[3]), 0, 4);
            const float sc = group_scale(sumsq, 1.0f / 64.0f);
            const float inv = rcp_rn(sc);
            // q = rne(x * inv): for a finite scale |q| <= 1016, and adding and
            // removing 1.5 * 2^23 rounds to the integer, ties to even, exactly
            // in fp16 (quant_pair_finite's integer); otherwise the saturating
            // conversion of the reference, as int16 converted to fp16
            uint32_t h[8];  // h[2v + e]: elements 16v + 4tj + 2e, +1
            if (__builtin_expect(__builtin_isfinite(sc), 1)) {
                constexpr float kMagic = 12582912.0f;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float r0 = (xv[v].x * inv + kMagic) - kMagic, r1 = (xv[v].y * inv + kMagic) - kMagic;
                    const float r2 = (xv[v].z * inv + kMagic) - kMagic, r3 = (xv[v].w * inv + kMagic) - kMagic;
                    h[2 * v] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r0, r1));
                    h[2 * v + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r2, r3));
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t q0 = quant_pair(xv[v].x * inv, xv[v].y * inv);
                    const uint32_t q1 = quant_pair(xv[v].z * inv, xv[v].w * inv);
                    h[2 * v] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(
                                                      (float)(int16_t)(q0 & 0xFFFF), (float)(int16_t)(q0 >> 16)));
                    h[2 * v + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(
                                                          (float)(int16_t)(q1 & 0xFFFF), (float)(int16_t)(q1 >> 16)));
                }
            }
            // elements 16v + 4tj + c are halves 4(tj % 2) + c of piece 2v + tj / 2,
            // i.e. (u, lane c') = (tj / 2, 16v + m)
            unsigned char *Ab = reinterpret_cast<unsigned char *>(Al);
#pragma unroll
            for (int v = 0; v < 4; ++v)
                *reinterpret_cast<uint2 *>(Ab + ((g * 2 + (tj >> 1)) * 64 + 16 * v + m) * 16 + 8 * (tj & 1)) =
                    real ? make_uint2(h[2 * v], h[2 * v + 1]) : make_uint2(0u, 0u);
            if (tj == 0) asl[g * 16 + m] = real ? sc : 0.0f;
        }
    };
    // the first batch straight-line: its loads went out before the weight
    // ring's, and this code's wait for them leaves the ring in flight
    quant_batch(0);
    for (int tb = QB * (NT / 4); tb < nteam; tb += QB * (NT / 4)) {
        load_batch(tb);
        quant_batch(tb);
    }
    __syncthreads();
    if (nq == 0) {  // no tile for this wave: an empty partial (no barrier follows)
        if (part_val && (lane & 15) == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * (lane >> 4) + i < M) {
                    part_val[(size_t)gw * M + 4 * (lane >> 4) + i] = -FLT_MAX;
                    part_idx[(size_t)gw * M + 4 * (lane >> 4) + i] = -1;
                }
        }
        return;
    }

    float4 out = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float bv[4] = {-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
    int32_t bi[4] = {-1, -1, -1, -1};
    auto step = [&](int sl, int Q) __attribute__((always_inline)) {
        const int g0 = 4 * (Q % qpt);
        half8_t bf[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const u32x4 v = wr[sl][u];
            uint32_t w[8];
            widen4_mf(v.x, w[0], w[1]);
            widen4_mf(v.y, w[2], w[3]);
            widen4_mf(v.z, w[4], w[5]);
            widen4_mf(v.w, w[6], w[7]);
            bf[u][0] = __builtin_bit_cast(half8_t, (u32x4){w[0], w[1], w[2], w[3]});
            bf[u][1] = __builtin_bit_cast(half8_t, (u32x4){w[4], w[5], w[6], w[7]});
        }
        // the scales copied out by real moves: kept as the slot's registers,
        // they would be live across the reload, which then takes other
        // registers and the loop's back edge copies them after a wait for
        // every load in flight
        float ws[4];
        asm volatile("v_mov_b32 %0, %1" : "=v"(ws[0]) : "v"(wsr[sl].x));
        asm volatile("v_mov_b32 %0, %1" : "=v"(ws[1]) : "v"(wsr[sl].y));
        asm volatile("v_mov_b32 %0, %1" : "=v"(ws[2]) : "v"(wsr[sl].z));
        asm volatile("v_mov_b32 %0, %1" : "=v"(ws[3]) : "v"(wsr[sl].w));
        // the slot's reload goes out here, after its values are consumed and
        // before this quad's MFMAs (pinned: left to itself, the scheduler
        // hoists reloads into fresh registers ahead of earlier uses, and the
        // ring's loads then retire in an order that makes each use wait for
        // nearly every load in flight)
        __builtin_amdgcn_sched_barrier(0);
        load(sl, min(Q + D, nq - 1));  // (past the last quad: the last again)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int g = g0 + u;
            const half8_t a0 = __builtin_bit_cast(half8_t, Al[(g * 2 + 0) * 64 + lane]);
            const half8_t a1 = __builtin_bit_cast(half8_t, Al[(g * 2 + 1) * 64 + lane]);
            const float4 as4 = *reinterpret_cast<const float4 *>(asl + g * 16 + 4 * c);
            float4_t acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, bf[u][0], (float4_t){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, bf[u][1], acc, 0, 0, 0);
            out.x = fmaf(acc[0] * as4.x, ws[u], out.x);
            out.y = fmaf(acc[1] * as4.y, ws[u], out.y);
            out.z = fmaf(acc[2] * as4.z, ws[u], out.z);
            out.w = fmaf(acc[3] * as4.w, ws[u], out.w);
        }
        if (Q % qpt == qpt - 1) {  // uniform: the tile's last quad
            const int col = 16 * (t0 + Q / qpt) + nl;
            const float o4[4] = {out.x, out.y, out.z, out.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 4 * c + i;
                if (row < M && col < N) {
                    if (C) C[(size_t)row * N + col] = o4[i];
                    if (o4[i] > -FLT_MAX) am_combine(bv[i], bi[i], o4[i], col);
                }
            }
            out = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    // nq is a multiple of D (D divides the quads of a tile): whole ring turns
    for (int Q0 = 0; Q0 < nq; Q0 += D) {
#pragma unroll
        for (int j = 0; j < D; ++j) step(j, Q0 + j);
    }
    // ---- the wave's partial per row: the 16 lanes of row group c
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
            const float ov = __shfl_xor(bv[i], off);
            const int32_t oi = __shfl_xor(bi[i], off);
            am_combine(bv[i], bi[i], ov, oi);
        }
        const int row = 4 * c + i;
        if (part_val && nl == 0 && row < M) {
            part_val[(size_t)gw * M + row] = bv[i];
            part_idx[(size_t)gw * M + row] = bi[i];
        }
    }
}

constexpr int kWideD = 2;   // quads in flight per wave of gemm_mf_wide_kernel
constexpr int kWideNW = 4;  // waves per block
constexpr int kWideBPC = 1; // blocks per CU

bool gemm_mf_wide_serves(int M, int N, int K) {
    // K: whole quads of groups, the ring's D quads dividing a tile's, and the
    // block's A fragments (32 K bytes) within half of a CU's LDS
    return M >= 1 && M <= 16 && N >= 16 && K > 0 && K % (256 * kWideD) == 0 && K <= 2048;
}

// Waves: kWideBPC blocks of kWideNW waves per CU, fewer where the weight has
// fewer 16-row tiles; one argmax partial each. (Fewer, longer waves measured
// faster than two blocks per CU: the blocks' prologue quantizers repeat the
// same work.)
int gemm_mf_wide_parts(int N, int cus) {
    const int ntiles = (N + 15) / 16;
    const int blocks = min(kWideBPC * max(cus, 1), (ntiles + kWideNW - 1) / kWideNW);
    return blocks * kWideNW;
}

hipError_t launch_gemm_mf_wide(const float *A, const int8_t *W, const float *S, float *C, int M, int N,
                               int K, float *part_val, int32_t *part_idx, int cus, hipStream_t st) {
    if (!gemm_mf_wide_serves(M, N, K) || (size_t)N * K > 0x7fffffffULL || (!part_val) != (!part_idx) ||
        (!C && !part_val))
        return hipErrorInvalidValue;
    const int ntiles = (N + 15) / 16, nwaves = gemm_mf_wide_parts(N, cus);
    const size_t lds = (size_t)(K / 64) * (2 * 64 * 16 + 16 * 4);
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void *>(&gemm_mf_wide_kernel<kWideD, kWideNW, 2>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)((2048 / 64) * (2 * 64 * 16 + 16 * 4)));
    if (attr != hipSuccess) return attr;
    gemm_mf_wide_kernel<kWideD, kWideNW, 2><<<nwaves / kWideNW, 64 * kWideNW, lds, st>>>(
        A, W, S, N, K, M, nwaves, ntiles, C, part_val, part_idx);
    return hipGetLastError();
}

}  // namespace q3vl
