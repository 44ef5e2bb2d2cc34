// gemm_skinny.hip -- 2..16 activation rows against an int8 weight at group
// size 64 or 128 (gfx950): the linears of a small decode batch.
//
// Reference: the general path of linear_int8_fp32s_int32acc_transpose,
// matmul/src/cpu_f32a_i8f32sb_f32c_avx2.cpp:477-662 (see gemm_t16.hip): G
// exact per group by fp16 MFMA, acc = fma(float(G) * a_s, w_s, acc) over the
// groups in ascending order.
//
// So few rows give one 16 x 16 output tile per 16 weight rows: 128 tiles at N =
// 2048, half the CUs, and one wave walking a tile's 96 groups (K = 6144) would
// take its loads' latency over and over. Here a block of 8 waves takes one
// tile and splits its K: wave w loads, widens and multiplies the 128-byte
// pieces w, w + 8, ... of the 16 weight rows, all of whose loads go out at
// once, and leaves the products t = G * a_s of its groups in LDS; then the
// threads, one an output, run the ordered sums acc = fma(t, w_s, acc) over all
// groups. The products and the sum round where the reference rounds, so
// splitting them over waves changes no bit.
// * Weights: 8 rows by 128 bytes a load (8 consecutive lanes a row; the MFMA's
//   own order of 16 rows by 64 bytes costs the vector cache six times as
//   much), through LDS with 16-byte pieces at slot piece ^ (row / 2), so that
//   a fragment read meets 16 bank groups. The products of a piece's groups
//   take its place.
// * Measured (graph replay, weights rotating; the integer GEMV that ran 2..8
//   rows and the 32-row GEMM that ran 9..16 before it in brackets): 4 x 2048 x
//   2048 4.2 us [7.7], 4 x 6144 x 2048 5.7 [10.2], 8 x 4096 x 4096 8.9 [18.1],
//   16 x 2048 x 2048 6.3 [18.8], 16 x 2048 x 6144 12.7 with its quantizer
//   launch [46.4]. What is left is one latency chain: the launch, the loads,
//   the quantizer or the weights' LDS pass, the ordered sums.
// * Activations: either fp32, quantized by the wave that needs them (a quad of
//   lanes a row and group, as quantize_t16_kernel; no launch for it), or the
//   fragments of quantize_t16_kernel.
#include "q3vl_device.hpp"
#include "q3vl_kernels.hpp"
#include "q3vl_mfma.hpp"

namespace q3vl {

// NP: 128-byte pieces per wave. RW: rows the quantizer pads to (4, 8 or 16);
// 0: the activations come as fragments. SW: segments 0 and 1 are gate and up
// weights and the block takes a column tile of each, half of its threads
// summing either; H = silu(gate) * up goes to segment 0's C.
template <int GS, int NP, int RW, bool SW>
__global__ __launch_bounds__(512) void gemm_skinny_kernel(GemmSkinnyArgs a) {
    constexpr int NW = 8, GP = 128 / GS;    // waves; groups of a piece
    constexpr int NT = SW ? 2 : 1;          // weight tiles
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, nl = lane & 15;
    const int K = a.K, Kg = K / GS, np = K / 128;
    // the block's segment and columns
    int tile = blockIdx.x, sg = 0;
    if (!SW)
        while (sg + 1 < a.nseg && tile >= (a.seg[sg].N + 15) / 16) tile -= (a.seg[sg++].N + 15) / 16;
    const int N = a.seg[sg].N, n0 = 16 * tile;

    unsigned char *wl = smem;                                              // [NT][np][2 KB]
    float *sl = reinterpret_cast<float *>(smem + NT * np * 2048);          // [NT][Kg][16]
    unsigned char *al = smem + NT * (np * 2048 + Kg * 64);                        // [np][2 chunks][2][4 RW pieces]
    float *asl = reinterpret_cast<float *>(al + (RW ? (size_t)np * 256 * RW : 0));  // [Kg][16]

    // ---- loads, oldest first what is used first: w_s, activations, weights
    // (pieces past the row's end repeat its last one and are not used)
    constexpr int SN = (NP * NW * GP * 16 + 511) / 512;
    float sreg[NT][SN];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < SN; ++i) {  // (row, group): groups fastest
            const int p = tid + 512 * i, r = p / Kg, g = p % Kg;
            sreg[t][i] = a.seg[sg + t].S[(size_t)min(n0 + min(r, 15), N - 1) * Kg + g];
        }
    constexpr int IT = RW ? (RW * NP * GP + 15) / 16 : 1;  // passes of the quantizer's 16 teams
    constexpr int QB = IT < 4 ? IT : 4;                    // passes whose loads are in flight
    float4 xb[QB][GS / 16];
    const int tj = lane & 3, team = lane >> 2;
    // item: row and group-in-wave of pass it; pieces of the wave: wid + 8 i
    auto item = [&](int it, int &m, int &gi, bool &in) __attribute__((always_inline)) {
        const int x = it * 16 + team;
        m = x % (RW ? RW : 1);
        gi = x / (RW ? RW : 1);
        in = gi < NP * GP && wid + NW * (gi / GP) < np;
    };
    auto load_x = [&](int it0) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < QB; ++it) {
            int m, gi;
            bool in;
            item(it0 + it, m, gi, in);
            const int g = min((wid + NW * (gi / GP)) * GP + gi % GP, Kg - 1);
            const float *x = a.A + (size_t)min(m, a.M - 1) * K + (size_t)g * GS + 4 * tj;
#pragma unroll
            for (int v = 0; v < GS / 16; ++v) xb[it][v] = *reinterpret_cast<const float4 *>(x + 16 * v);
        }
    };
    if constexpr (RW > 0) load_x(0);
    u32x4 fr[NP][4];       // fragments: [piece][chunk][MFMA]
    float4 as4[NP][GP];
    if constexpr (RW == 0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = min(wid + NW * i, np - 1);
#pragma unroll
            for (int x = 0; x < 4; ++x)
                fr[i][x] = reinterpret_cast<const u32x4 *>(a.Af)[((size_t)(2 * p + (x >> 1)) * 4 + (x & 1)) * 64 + lane];
#pragma unroll
            for (int g = 0; g < GP; ++g)
                as4[i][g] = *reinterpret_cast<const float4 *>(a.asf + (size_t)(p * GP + g) * 32 + c * 8);
        }
    }
    u32x4 wr[NT][NP][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = min(wid + NW * i, np - 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = 8 * h + (lane >> 3);
                wr[t][i][h] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(
                    a.seg[sg + t].W + (size_t)min(n0 + r, N - 1) * K + p * 128 + 16 * ((lane & 7) ^ ((r >> 1) & 7))));
            }
        }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < SN; ++i) {
            const int p = tid + 512 * i, r = p / Kg, g = p % Kg;
            if (r < 16) sl[(t * Kg + g) * 16 + r] = sreg[t][i];
        }
    // ---- quantize the wave's groups
    if constexpr (RW > 0) {
#pragma unroll
        for (int it0 = 0; it0 < IT; it0 += QB) {
            if (it0 > 0) load_x(it0);
#pragma unroll
            for (int it = 0; it < QB; ++it) {
                if (it0 + it >= IT) break;
                int m, gi;
                bool in;
                item(it0 + it, m, gi, in);
                const int p = wid + NW * (gi / GP);
                const float s = quant_team<GS>(xb[it], [&](int v, uint32_t h0, uint32_t h1) {
                    // elements 16v + 4tj of the group: the k = e.. of chunk e / 64 -> (u, lane group) as the weights' bytes
                    const int e = (gi % GP) * GS + 16 * v + 4 * tj;
                    const int ch = e >> 6, u = (e >> 3) & 1, cc = (e & 63) >> 4;
                    if (in)
                        *reinterpret_cast<uint2 *>(al + ((size_t)(p * 2 + ch) * 2 + u) * (64 * RW) + (cc * RW + m) * 16 +
                                                   (e & 7) * 2) = make_uint2(h0, h1);
                });
                if (in && tj == 0) asl[(p * GP + gi % GP) * 16 + m] = s;
            }
        }
    }
    // ---- weights through LDS (the wave's own region: no barrier)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = wid + NW * i;
            if (p < np) {  // uniform
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<u32x4 *>(wl + (t * np + p) * 2048 + h * 1024 + lane * 16) = wr[t][i][h];
            }
        }
    wave_lds_sync();  // rows, scales and weights that other lanes wrote
#pragma unroll
    for (int ti = 0; ti < NT * NP; ++ti) {
        const int i = ti % NP, p = wid + NW * i;
        unsigned char *wp = wl + (ti / NP * np + p) * 2048;
        if (p < np) {  // uniform
            u32x4 raw[2];
#pragma unroll
            for (int ch = 0; ch < 2; ++ch)
                raw[ch] = *reinterpret_cast<const u32x4 *>(wp + nl * 128 + (((4 * ch + c) ^ (nl >> 1)) & 7) * 16);
            wave_lds_sync();  // the products take the place of what every lane has read
            float4_t acc[GP];
#pragma unroll
            for (int ch = 0; ch < 2; ++ch) {
                const int g = GP == 2 ? ch : 0;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    u32x4 av;
                    if constexpr (RW > 0)
                        av = *reinterpret_cast<const u32x4 *>(al + ((size_t)(p * 2 + ch) * 2 + u) * (64 * RW) + (c * RW + nl % RW) * 16);
                    else
                        av = fr[i][2 * ch + u];
                    acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8_t, av), widen8(raw[ch][2 * u], raw[ch][2 * u + 1]),
                        (u == 0 && (GP == 2 || ch == 0)) ? (float4_t){0.0f, 0.0f, 0.0f, 0.0f} : acc[g], 0, 0, 0);
                }
            }
#pragma unroll
            for (int g = 0; g < GP; ++g) {
                // this lane's rows 4c .. 4c + 3 (rows past M hold a repeat or padding and are not kept)
                float4 s4;
                if constexpr (RW > 0) s4 = *reinterpret_cast<const float4 *>(asl + (p * GP + g) * 16 + (RW >= 16 ? 4 * c : 4 * (c % (RW / 4))));
                else s4 = as4[i][g];
                *reinterpret_cast<float4 *>(wp + g * 1024 + lane * 16) =
                    make_float4(acc[g][0] * s4.x, acc[g][1] * s4.y, acc[g][2] * s4.z, acc[g][3] * s4.w);
            }
        }
    }
    __syncthreads();
    // ---- the ordered sums: thread x = tid % 256 holds row 4 (x / 64) + x % 4,
    // column x / 4 % 16; SW: the upper 256 threads the up tile
    const int x = tid & 255, tt = SW ? tid >> 8 : 0;
    const int row = 4 * (x >> 6) + (x & 3), col = (x >> 2) & 15;
    float acc = 0.0f;
    if (row < a.M && (SW || tid < 256)) {
        const float *tp = reinterpret_cast<const float *>(wl + tt * np * 2048) + x;
        constexpr int TS = GS == 64 ? 256 : 512;  // floats from one group's products to the next
        const float *sp = sl + tt * Kg * 16 + col;
        int g = 0;
        for (; g + 16 <= Kg; g += 16) {
            float t[16], w[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                t[k] = tp[(g + k) * TS];
                w[k] = sp[(g + k) * 16];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) acc = fmaf(t[k], w[k], acc);
        }
        for (; g < Kg; ++g) acc = fmaf(tp[g * TS], sp[g * 16], acc);
    }
    if constexpr (SW) {
        __syncthreads();  // the products are read
        float *up = reinterpret_cast<float *>(smem);
        if (tt) up[x] = acc;
        __syncthreads();
        if (!tt && row < a.M && n0 + col < N) a.seg[0].C[(size_t)row * N + n0 + col] = silu_mul(acc, up[x]);
    } else if (tid < 256 && row < a.M && n0 + col < N) {
        a.seg[sg].C[(size_t)row * N + n0 + col] = acc;
    }
}

// Rows the quantizer pads to (0: fragments), and the 128-byte pieces a wave
// takes at most: what fits the LDS at every group size. One table for what is
// served and for the kernels there are.
static int skinny_rw(int M, bool fp32) { return !fp32 ? 0 : M <= 4 ? 4 : M <= 8 ? 8 : 16; }
static constexpr int skinny_pieces(int rw, bool swiglu) { return swiglu || rw == 16 ? 3 : rw == 8 ? 4 : 6; }

// LDS of a block: weights (then products), w_s, and the quantized rows.
static constexpr size_t skinny_lds(int rw, int K, int gs, bool swiglu) {
    const size_t kg = K / gs;
    return (swiglu ? 2 : 1) * ((size_t)K * 16 + kg * 64) + (rw ? (size_t)2 * K * rw + kg * 64 : 0);
}

template <int GS, int NP, int RW, bool SW> static hipError_t launch_one(const GemmSkinnyArgs &a, int grid, hipStream_t st) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_skinny_kernel<GS, NP, RW, SW>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess) return attr;
    gemm_skinny_kernel<GS, NP, RW, SW><<<grid, 512, skinny_lds(RW, a.K, GS, SW), st>>>(a);
    return hipGetLastError();
}

template <int GS, int RW, bool SW, int NP = skinny_pieces(RW, SW)>
static hipError_t launch_np(const GemmSkinnyArgs &a, int grid, hipStream_t st) {
    static_assert(skinny_lds(RW, 1024 * NP, GS, SW) <= 160 * 1024, "LDS");
    if constexpr (NP > 0) {
        if ((a.K / 128 + 7) / 8 == NP) return launch_one<GS, NP, RW, SW>(a, grid, st);
        return launch_np<GS, RW, SW, NP - 1>(a, grid, st);
    }
    return hipErrorInvalidValue;
}

template <int GS> static hipError_t launch_rw(const GemmSkinnyArgs &a, bool swiglu, int grid, hipStream_t st) {
    if (swiglu) return a.M <= 4 ? launch_np<GS, 4, true>(a, grid, st) : launch_np<GS, 8, true>(a, grid, st);
    if (!a.A) return launch_np<GS, 0, false>(a, grid, st);
    if (a.M <= 4) return launch_np<GS, 4, false>(a, grid, st);
    if (a.M <= 8) return launch_np<GS, 8, false>(a, grid, st);
    return launch_np<GS, 16, false>(a, grid, st);
}

bool gemm_skinny_serves(int M, int K, int gs, bool fp32, bool swiglu) {
    return M >= 2 && M <= (swiglu ? 8 : 16) && (gs == 64 || gs == 128) && K > 0 && K % 128 == 0 && (fp32 || !swiglu) &&
           K <= 1024 * skinny_pieces(skinny_rw(M, fp32), swiglu);
}

int gemm_skinny_per_cu(int M, int K, int gs, bool fp32, bool swiglu) {
    return (int)((160 * 1024) / skinny_lds(skinny_rw(M, fp32), K, gs, swiglu));
}

hipError_t launch_gemm_skinny(const GemmSkinnyArgs &a, int gs, bool swiglu, hipStream_t st) {
    if (!gemm_skinny_serves(a.M, a.K, gs, a.A != nullptr, swiglu) || a.nseg < 1 || a.nseg > 3 || (swiglu && a.nseg != 2) ||
        (!a.A && (!a.Af || !a.asf)))
        return hipErrorInvalidValue;
    int grid = 0;
    for (int i = 0; i < (swiglu ? 1 : a.nseg); ++i) grid += (a.seg[i].N + 15) / 16;
    if (grid == 0) return hipSuccess;
    return gs == 64 ? launch_rw<64>(a, swiglu, grid, st) : launch_rw<128>(a, swiglu, grid, st);
}

}  // namespace q3vl
