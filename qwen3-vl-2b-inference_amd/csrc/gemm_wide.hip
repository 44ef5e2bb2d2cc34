// gemm_wide.hip -- 2..16 activation rows against a very wide weight (the
// lm_head over a batch of rows), on 16x16x32 fp16 MFMA tiles (gfx950).
//
// Reference: the general path of linear_int8_fp32s_int32acc_transpose,
// matmul/src/cpu_f32a_i8f32sb_f32c_avx2.cpp:477-662 (see gemm_t16.hip), and
// greedy_decode (tokenizer/src/utils.cpp:34-44) for the argmax.
//
// The product is 16 rows x N with N * K of hundreds of MB: bound by reading
// the weights once. Per 16 x 16 tile and group of 64 a wave spends about 35
// issue slots (widening the weights is half of them), 19 us over the lm_head
// [151936, 2048], beside 52 us of reading; what used to hold it back was the
// vector cache (a load in the MFMA's lane order, 16 rows by 64 bytes, costs it
// ~94 cycles: 46 us a CU for the lm_head). So:
// * a wave walks a run of 16-row tiles, 256 bytes of each row (a "pair" of
//   128-byte lines) at a time, reaching LDS by loads with an LDS destination
//   that cover 4 rows x 256 bytes each, a ring of pairs ahead (wave-private:
//   no barrier), waited for by count. Slot s of row r holds piece s ^ r, so a
//   fragment read meets 16 bank groups.
// * The block quantizes the activations itself into LDS, as the fragments, a
//   quad of lanes a row and group, while the first pairs are on their way.
// * G of a group is the MFMAs' exact integer sum; lane l holds rows 4 (l / 16)
//   + i, column l % 16, and folds out = fma(G * a_s, w_s, out) in ascending
//   order. Per tile the wave keeps the greedy-argmax candidate of each row
//   (am_combine; values not above -FLT_MAX never win), at the end the block
//   one partial a row.
// * Measured, lm_head [151936, 2048] + argmax with the logits stored, us a
//   call, before in brackets: group 64, 2 rows 60.6 [65.8], 4 rows 62.2 [79.6],
//   8 rows 65.1 [77.7], 16 rows 66.1 [82.2]; group 32, 8 rows 67.8 [147], 16
//   rows 70.9 [250]; group 128, 8 rows 61.5 [119], 16 rows 62.7 [190]. The
//   kernel alone at 2 rows reads at 6.0 TB/s. Nontemporal weight loads: 74.9
//   -> 72.6 us at 8 rows; the logits four tiles at a time: 72.4 -> 65.5.
#include "q3vl_device.hpp"
#include "q3vl_kernels.hpp"
#include "q3vl_mfma.hpp"

namespace q3vl {

// RW: rows the activations are padded to (4, 8 or 16). NB: pairs in a wave's
// ring.
template <int GS, int RW, int NB>
__global__ __launch_bounds__(512) void gemm_wide_kernel(const float *A, const int8_t *W, const float *S, int N,
                                                        int K, int M, int nwaves, int ntiles, float *C,
                                                        float *part_val, int32_t *part_idx) {
    constexpr int NW = 8;
    constexpr int GP = 256 / GS;                       // groups of a pair
    constexpr int SI = GP * 16 <= 64 ? 1 : GP / 4;     // w_s loads of a pair
    constexpr int PAIR = 4096 + SI * 256;              // bytes of a ring slot: weights, w_s [row][GP]
    constexpr int LOADS = 4 + SI;                      // loads of a pair
    extern __shared__ __align__(16) unsigned char smem[];
    const int Kg = K / GS, np = K / 256;  // groups; pairs of a row
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, nl = lane & 15;
    const int gw = (int)blockIdx.x * NW + wid;
    // tiles [t0, t1): the waves' shares differ by at most one tile
    const int t0 = __builtin_amdgcn_readfirstlane((int)((long)gw * ntiles / nwaves));
    const int t1 = __builtin_amdgcn_readfirstlane((int)((long)(gw + 1) * ntiles / nwaves));
    const int nq = (t1 - t0) * np;  // pairs over the wave's tiles

    const int ring = wid * NB * PAIR;
    unsigned char *al = smem + NW * NB * PAIR;  // [chunk][2][4 RW pieces]
    float *asl = reinterpret_cast<float *>(al + (size_t)K * 2 * RW);  // [Kg][16]

    // resources at the wave's first row
    const int row0 = min(16 * t0, N - 1);
    const rsrc_t rW = make_rsrc(W + (size_t)row0 * K, (uint32_t)(N - row0) * K);
    const rsrc_t rS = make_rsrc(S + (size_t)row0 * Kg, (uint32_t)(N - row0) * Kg * 4);
    // the next pair of the wave's (lt, lp: its tile and place in the row;
    // past the last one it repeats, so that the count of loads in flight is
    // the same throughout)
    int lt = 0, lp = 0;
    int woff[4], soff[SI];
    const int nt = t1 - t0;
    auto rows_of = [&]() __attribute__((always_inline)) {  // tile lt's rows (clamped into the weight)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * i + (lane >> 4);
            woff[i] = (min(row0 + 16 * lt + r, N - 1) - row0) * K + 16 * ((lane & 15) ^ r);
        }
#pragma unroll
        for (int i = 0; i < SI; ++i) {
            const int x = (lane + 64 * i) % (16 * GP), r = x / GP;
            soff[i] = ((min(row0 + 16 * lt + r, N - 1) - row0) * Kg + x % GP) * 4;
        }
    };
    rows_of();
    auto load_pair = [&](int sl) __attribute__((always_inline)) {
        const int base = ring + sl * PAIR;
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16_nt(rW, woff[i], lp * 256, base + i * 1024);
#pragma unroll
        for (int i = 0; i < SI; ++i) dma4(rS, soff[i], lp * GP * 4, base + 4096 + i * 256);
        if (lp + 1 < np) ++lp;
        else if (lt + 1 < nt) {
            ++lt;
            lp = 0;
            rows_of();
        }
    };
    if (nq > 0) {
#pragma unroll
        for (int j = 0; j < NB; ++j) load_pair(j);
    }
    // ---- quantize the activations into LDS: items (row, group), rows fastest
    {
        const int tj = lane & 3, nitem = RW * Kg;
        for (int it = tid >> 2; it < nitem; it += 128) {  // whole quads
            const int m = it % RW, g = it / RW;
            const float *x = A + (size_t)min(m, M - 1) * K + (size_t)g * GS + 4 * tj;
            float4 cv[GS / 16];
#pragma unroll
            for (int v = 0; v < GS / 16; ++v) cv[v] = *reinterpret_cast<const float4 *>(x + 16 * v);
            const float s = quant_team<GS>(cv, [&](int v, uint32_t h0, uint32_t h1) {
                const int k = g * GS + 16 * v + 4 * tj, e = k & 63;
                const int cc = GS == 32 ? (e >> 3) & 3 : e >> 4, u = GS == 32 ? e >> 5 : (e >> 3) & 1;
                *reinterpret_cast<uint2 *>(al + ((size_t)(k >> 6) * 2 + u) * (64 * RW) + (cc * RW + m) * 16 + (e & 7) * 2) =
                    make_uint2(h0, h1);
            });
            if (tj == 0) asl[g * 16 + m] = s;
        }
    }
    dma_wait<0>();
    __syncthreads();

    float4_t out = {0.0f, 0.0f, 0.0f, 0.0f};
    const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float bv[4] = {-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
    int32_t bi[4] = {-1, -1, -1, -1};
    int sl = 0, p = 0, tl = 0;  // ring slot, pair of the row, tile of the run
    // the logits of four tiles together go out through the ring slot that the
    // last of them has emptied, 256 bytes a row (one by one, 64 bytes a row:
    // 72.4 against 67.5 us for 8 rows of the lm_head)
    float4 kept[4];
    const bool vec = C && N % 4 == 0 && ((uintptr_t)C & 15) == 0;  // 16-byte stores
    for (int Q = 0; Q < nq; ++Q) {
        dma_wait<LOADS *(NB - 1)>();
        const unsigned char *rb = smem + ring + sl * PAIR;
        // the pair to registers; then its slot takes the pair NB further on
        u32x4 raw[4];
        float ws[GP];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (GS == 32) {  // 8 bytes of each of the chunk's two groups
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 g0 = *reinterpret_cast<const u32x2 *>(rb + nl * 256 + ((4 * u + (c >> 1)) ^ nl) * 16 + 8 * (c & 1));
                const u32x2 g1 = *reinterpret_cast<const u32x2 *>(rb + nl * 256 + ((4 * u + 2 + (c >> 1)) ^ nl) * 16 + 8 * (c & 1));
                raw[u] = (u32x4){g0[0], g0[1], g1[0], g1[1]};
            } else {
                raw[u] = *reinterpret_cast<const u32x4 *>(rb + nl * 256 + ((4 * u + c) ^ nl) * 16);
            }
        }
#pragma unroll
        for (int g = 0; g < GP; ++g) ws[g] = reinterpret_cast<const float *>(rb + 4096)[nl * GP + g];
        half8_t bf[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            bf[u][0] = widen8(raw[u][0], raw[u][1]);
            bf[u][1] = widen8(raw[u][2], raw[u][3]);
        }
#pragma unroll
        for (int g = 0; g < GP; ++g) asm volatile("" : "+v"(ws[g]));  // (read before the slot is reloaded)
        __builtin_amdgcn_sched_barrier(0);
        // (after the fourth tile's last pair the logits pass through the slot first)
        const bool flush = vec && p + 1 == np && (tl & 3) == 3 && row0 + 16 * (tl + 1) <= N;
        if (!flush) load_pair(sl);
        __builtin_amdgcn_sched_barrier(0);
        float4_t acc[GP];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const half8_t av = __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4 *>(
                    al + ((size_t)(p * 4 + u) * 2 + k) * (64 * RW) + (c * RW + nl % RW) * 16));
                const int g = GS == 32 ? 2 * u + k : GS == 64 ? u : u >> 1;
                const bool first = GS == 32 || (k == 0 && (GS == 64 || (u & 1) == 0));
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bf[u][k], first ? zero : acc[g], 0, 0, 0);
            }
#pragma unroll
        for (int g = 0; g < GP; ++g) {
            const float4 as4 = *reinterpret_cast<const float4 *>(asl + (p * GP + g) * 16 + 4 * (RW == 16 ? c : c % (RW / 4)));
            out[0] = fmaf(acc[g][0] * as4.x, ws[g], out[0]);
            out[1] = fmaf(acc[g][1] * as4.y, ws[g], out[1]);
            out[2] = fmaf(acc[g][2] * as4.z, ws[g], out[2]);
            out[3] = fmaf(acc[g][3] * as4.w, ws[g], out[3]);
        }
        if (++p == np) {  // uniform: the tile's last pair
            const int col = row0 + 16 * tl + nl, j4 = tl & 3;
            // one of four tiles that leave together?
            const bool four = vec && (tl | 3) < nt && row0 + 16 * ((tl | 3) + 1) <= N;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 4 * c + i;
                if (row < M && col < N) {
                    if (out[i] > -FLT_MAX) am_combine(bv[i], bi[i], out[i], col);
                    if (C && !four) C[(size_t)row * N + col] = out[i];
                }
                kept[i].x = j4 == 0 ? out[i] : kept[i].x;
                kept[i].y = j4 == 1 ? out[i] : kept[i].y;
                kept[i].z = j4 == 2 ? out[i] : kept[i].z;
                kept[i].w = j4 == 3 ? out[i] : kept[i].w;
            }
            if (flush) {
                float *ot = reinterpret_cast<float *>(smem + ring + sl * PAIR);  // [16 rows][64]
                wave_lds_sync();
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float *d = ot + (4 * c + i) * 64 + nl;
                    d[0] = kept[i].x;
                    d[16] = kept[i].y;
                    d[32] = kept[i].z;
                    d[48] = kept[i].w;
                }
                wave_lds_sync();
#pragma unroll
                for (int q = 0; q < RW / 4; ++q) {
                    const int row = 4 * q + c;
                    const float4 v = *reinterpret_cast<const float4 *>(ot + row * 64 + 4 * nl);
                    if (row < M) *reinterpret_cast<float4 *>(C + (size_t)row * N + row0 + 16 * (tl - 3) + 4 * nl) = v;
                }
                wave_lds_sync();
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the slot is reloaded
                load_pair(sl);
            }
            out = zero;
            p = 0;
            ++tl;
        }
        sl = sl + 1 == NB ? 0 : sl + 1;
    }
    dma_wait<0>();  // (no load outlives the block)
    // ---- the block's partial per row: the 16 lanes of a row group, then the
    // waves through LDS (empty ones where a wave has no tile)
    if (!part_val) return;  // uniform
    __syncthreads();        // the ring is free
    float *rv = reinterpret_cast<float *>(smem);  // [NW][16]
    int32_t *ri = reinterpret_cast<int32_t *>(rv + NW * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
            const float ov = __shfl_xor(bv[i], off);
            const int32_t oi = __shfl_xor(bi[i], off);
            am_combine(bv[i], bi[i], ov, oi);
        }
        if (nl == 0) {
            rv[wid * 16 + 4 * c + i] = bv[i];
            ri[wid * 16 + 4 * c + i] = bi[i];
        }
    }
    __syncthreads();
    if (tid < M) {
        float v = -FLT_MAX;
        int32_t x = -1;
#pragma unroll
        for (int w = 0; w < NW; ++w) am_combine(v, x, rv[w * 16 + tid], ri[w * 16 + tid]);
        part_val[(size_t)blockIdx.x * M + tid] = v;
        part_idx[(size_t)blockIdx.x * M + tid] = x;
    }
}

static size_t wide_lds(int M, int K, int gs) {
    const size_t rw = M <= 4 ? 4 : M <= 8 ? 8 : 16, nb = M <= 8 ? 3 : 2;
    const size_t pair = 4096 + (gs == 32 ? 512 : 256);
    return 8 * nb * pair + (size_t)K * 2 * rw + (size_t)(K / gs) * 64;
}

bool gemm_wide_serves(int M, int N, int K, int gs) {
    return M >= 2 && M <= 16 && N >= 16 && (gs == 32 || gs == 64 || gs == 128) && K > 0 && K % 256 == 0 &&
           K <= (1 << 16) && wide_lds(M, K, gs) <= 160 * 1024;
}

// One block of 8 waves per CU, fewer where the weight has fewer 16-row tiles;
// one argmax partial a block. (Each block repeats the quantizer.)
int gemm_wide_parts(int N, int cus) { return min(max(cus, 1), ((N + 15) / 16 + 7) / 8); }

template <int GS, int RW, int NB>
static hipError_t launch_wide(const float *A, const int8_t *W, const float *S, float *C, int M, int N, int K,
                              float *part_val, int32_t *part_idx, int cus, hipStream_t st) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_wide_kernel<GS, RW, NB>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess) return attr;
    const int blocks = gemm_wide_parts(N, cus);
    gemm_wide_kernel<GS, RW, NB><<<blocks, 512, wide_lds(M, K, GS), st>>>(A, W, S, N, K, M, 8 * blocks, (N + 15) / 16, C,
                                                                        part_val, part_idx);
    return hipGetLastError();
}

hipError_t launch_gemm_wide(const float *A, const int8_t *W, const float *S, float *C, int M, int N, int K, int gs,
                            float *part_val, int32_t *part_idx, int cus, hipStream_t st) {
    if (!gemm_wide_serves(M, N, K, gs) || (size_t)N * K > 0x7fffffffULL || (!part_val) != (!part_idx) ||
        (!C && !part_val))
        return hipErrorInvalidValue;
#define Q3VL_WIDE(G)                                                                                       \
    if (gs == G)                                                                                           \
        return M <= 4 ? launch_wide<G, 4, 3>(A, W, S, C, M, N, K, part_val, part_idx, cus, st)             \
               : M <= 8 ? launch_wide<G, 8, 3>(A, W, S, C, M, N, K, part_val, part_idx, cus, st)           \
                        : launch_wide<G, 16, 2>(A, W, S, C, M, N, K, part_val, part_idx, cus, st);
    Q3VL_WIDE(32) Q3VL_WIDE(64) Q3VL_WIDE(128)
#undef Q3VL_WIDE
    return hipErrorInvalidValue;
}

}  // namespace q3vl
