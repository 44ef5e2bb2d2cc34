// gemm_t16.hip -- int8-weight GEMM for M > 8 at group sizes 32, 64 and 128
// (gfx950), on 16x16x32 fp16 MFMA tiles; weights and activations reach LDS by
// loads with an LDS destination, the weights are widened from there.
//
// Reference: the general path of linear_int8_fp32s_int32acc_transpose,
// matmul/src/cpu_f32a_i8f32sb_f32c_avx2.cpp:477-662: for each output and
// each K-group g in ascending order, G = sum_{k in g} q[m,k] * w[n,k] exactly
// (int32), then acc = fma(float(G) * a_s[m,g], w_s[n,g], acc) (:613-617,
// 652; GCC contracts the multiply-add, which the golden vectors pin).
//
// Exactness. q (int16, |q| <= 127 sqrt(128)) and w (int8) are exact in fp16,
// and every partial sum of one group is an integer below 2^24, so the MFMAs
// over the group's k with a zero initial accumulator yield G exactly. (A
// group whose scale is not finite holds q of 0 and -32768 only: its sums are
// multiples of 2^15 and exact as well.)
//
// What bounds it. Probes on MI355X at 2.4 GHz: a SIMD issues one fp32
// instruction of a wave every 4 to 5 cycles with two waves on it (5 to 8 with
// one), a 16x16x32 MFMA holds the vector pipe for about 9, and a wave's MFMAs
// and VALU work add up rather than overlap. A 16 x 16 output tile costs per
// group of 64 two MFMAs, 8 VALU operations of the fold (the reference rounds
// the product and the sum apart) and its share of widening the weights (16
// operations a 16-column tile, shared by the block's row tiles): about 25 ns
// a SIMD, and 29 to 36 measured in the loop. Counters: with two waves or more
// a SIMD and whole rounds of large tiles the two units together are busy three
// quarters of the time (1280 x 6144 x 2048 SwiGLU: VALU 49 %, MFMA 26 %), at
// 512 rows about two thirds; with one block a CU a half, and with one wave a
// SIMD a third (196 x 2048 x 4096: 22 and 9 %), the rest being the group's
// chain of LDS reads, MFMAs, scaling and folds, which too few waves hide. So
// the large products come near the issue limit and the small ones wait; for
// both, everything else is kept off the issue slots:
// * weights and activations reach LDS by loads with an LDS destination (no
//   registers, no LDS stores; 170 instead of 224 VGPRs at 128 x 256), waited
//   for by count;
// * a weight load covers whole 128-byte pieces of 8 rows. Read straight into
//   the MFMA's lane order (16 rows by 64 bytes) each load cost the vector
//   cache ~94 cycles instead of ~16: 512 x 2048 x 6144 34.4 -> 27.5 us;
// * the activation scales ride in one register per 64 rows and reach the
//   accumulator rows by DPP row broadcast inside the multiply;
// * fragments are read three row tiles ahead, MFMAs issued one tile ahead of
//   their fold.
#include <type_traits>

#include "q3vl_device.hpp"
#include "q3vl_kernels.hpp"
#include "q3vl_mfma.hpp"

namespace q3vl {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ------------------------------------------------------- activation fragments
// q in fp16, in chunks of 64 k: per 32-row m-tile t and chunk c a 4 KB block
// [16-row half][MFMA u][lane][8 halves], lane l holding row l % 16 and the k
// that its weight bytes hold: with c = l / 16, k = 16c + 8u + j at group
// sizes 64 and 128 (a lane's 16 weight bytes feed both MFMAs of the chunk),
// k = 32u + 8c + j at 32 (one group an MFMA). The scales come per m-tile and
// group as 32 floats [r][4 half + i] of row 16 half + 4r + i: what the 16
// lanes of DPP row r need for the accumulator rows they hold.
template <int GS>
Q3VL_INLINE size_t frag_off(int mt, int row32, int Kc, int k) {
    const int e = k & 63;
    const int c = GS == 32 ? (e >> 3) & 3 : e >> 4, u = GS == 32 ? e >> 5 : (e >> 3) & 1;
    return (((((size_t)mt * Kc + (k >> 6)) * 2 + (row32 >> 4)) * 2 + u) * 64 + (row32 & 15) + 16 * c) * 16 +
           (e & 7) * 2;
}
Q3VL_INLINE size_t frag_scale(int mt, int row32, int Kg, int g) {
    return ((size_t)mt * Kg + g) * 32 + ((row32 >> 2) & 3) * 8 + 4 * (row32 >> 4) + (row32 & 3);
}

// A block of 128 threads takes 8 rows x 4 groups: a 128-byte line of the
// fragment order holds 16 bytes of 8 consecutive rows, so every line is
// written whole by one block.
template <int GS>
__global__ __launch_bounds__(128) void quantize_t16_kernel(const float *__restrict__ A,
                                                           unsigned char *__restrict__ qf,
                                                           float *__restrict__ asf, int M, int K) {
    const int Kg = K / GS, Kc = K / 64;
    const int j = threadIdx.x & 3, team = threadIdx.x >> 2;
    const int g = blockIdx.x * 4 + (team & 3), m = blockIdx.y * 8 + (team >> 2);
    if (g >= Kg) return;  // whole quads leave together
    const bool real = m < M;
    float4 cv[GS / 16];
    const float *x = A + (size_t)(real ? m : M - 1) * K + (size_t)g * GS + 4 * j;
#pragma unroll
    for (int v = 0; v < GS / 16; ++v) {
        const float4 f = *reinterpret_cast<const float4 *>(x + 16 * v);
        cv[v] = real ? f : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    const float s = quant_team<GS>(cv, [&](int v, uint32_t h0, uint32_t h1) {
        *reinterpret_cast<uint2 *>(qf + frag_off<GS>(m >> 5, m & 31, Kc, g * GS + 16 * v + 4 * j)) =
            real ? make_uint2(h0, h1) : make_uint2(0u, 0u);
    });
    if (j == 0) asf[frag_scale(m >> 5, m & 31, Kg, g)] = real ? s : 0.0f;
}

hipError_t launch_quantize_t16(const float *A, _Float16 *qf, float *asf, int M, int K, int gs,
                               hipStream_t st) {
    if (K % 64 != 0 || M < 1) return hipErrorInvalidValue;
    const dim3 grid((K / gs + 3) / 4, (M + 31) / 32 * 4);
    unsigned char *q = reinterpret_cast<unsigned char *>(qf);
    if (gs == 32) quantize_t16_kernel<32><<<grid, 128, 0, st>>>(A, q, asf, M, K);
    else if (gs == 64) quantize_t16_kernel<64><<<grid, 128, 0, st>>>(A, q, asf, M, K);
    else if (gs == 128) quantize_t16_kernel<128><<<grid, 128, 0, st>>>(A, q, asf, M, K);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---------------------------------------------------------------- the GEMM
// The tile shape. GS: group size. A: 16-row tiles of the block (2, 4 or 8:
// all of its waves share its rows). B: 16-column tiles of a wave (SwiGLU: B/2
// gate, B/2 up). NW: waves, side by side along the columns. A unit is UC
// chunks of 64 k: one group of 64 or 128, two of 32. SU: units of a stage of
// activations (three in LDS). NB: stages of weights (128 bytes of each row)
// in LDS per wave.
template <int GS_, int A_, int B_, int NW_, int SU_, int NB_, bool SWIGLU_> struct T16 {
    static constexpr int GS = GS_, A = A_, B = B_, NW = NW_, SU = SU_, NB = NB_;
    static constexpr bool SWIGLU = SWIGLU_;
    static constexpr int NT = 64 * NW;               // threads
    static constexpr int NJ = SWIGLU ? B / 2 : B;    // output column tiles of a wave
    static constexpr int COLS = 16 * NW * NJ;        // output columns of the block
    static constexpr int MT = A / 2;                 // 32-row m-tiles of the block
    static constexpr int UC = GS == 128 ? 2 : 1;     // chunks of a unit
    static constexpr int GU = GS == 32 ? 2 : 1;      // groups of a unit
    static constexpr int UB = 2 / UC;                // units of a weight stage
    static constexpr int NM = 2 * UC;                // MFMAs of a tile and unit
    static constexpr int SC = SU * UC, SG = SU * GU; // chunks, groups of an activation stage
    static constexpr int NG = 4 * GU;                // groups of the loop body (four units)
    static constexpr int PD = 3;                     // steps that fragments are read ahead
    static constexpr int CB = (A - 1 + PD) / A;      // units before the next stage that first read it
    static constexpr int ABUF = MT * SC * 4096;      // bytes of a stage's fragments
    static constexpr int NA = ABUF / 1024 / NW;      // loads per wave and stage
    static constexpr int SBYTES = MT * SG * 128;     // bytes of a stage's scales
    static constexpr int SBUF = (SBYTES + 1023) / 1024 * 1024;
    static constexpr int WST = NG / 4;               // w_s loads per column tile and body
    static constexpr int OFF_S = 3 * ABUF, OFF_B = OFF_S + 3 * SBUF;
    static constexpr int OFF_W = OFF_B + NW * B * NB * 2048, LDS = OFF_W + NW * 2 * B * WST * 256;
    static_assert(A == 2 || A == 4 || A == 8, "rows");
    static_assert(!SWIGLU || B % 2 == 0, "gate and up tiles");
    static_assert(SU >= CB && 4 % SU == 0 && NA * 1024 * NW == ABUF && SBUF <= 1024 * NW, "stages");
    static_assert(LDS <= 160 * 1024, "LDS");
    // Which loads go out in unit u of the K loop (before its first unit: as
    // units -8 .. -1 would issue them, for the stages there are): the next
    // stage but one of the activations where unit u first reads the next, the
    // next body but one's w_s in a body's first unit (after the wait for the
    // weights), the weight stage that takes the slot consumed at the unit's
    // end. Stages below 0: none.
    static constexpr int fdiv(int a, int b) { return (a + 64 * b) / b - 64; }
    static constexpr int a_stage(int u) { return (u + 64) % SU == SU - CB ? fdiv(u, SU) + 2 : -1; }
    static constexpr int w_body(int u) { return (u + 64) % 4 == 0 ? fdiv(u, 4) + 2 : -1; }
    static constexpr int b_stage(int u) { return (u + 65) % UB == UB - 1 ? fdiv(u + 1, UB) + NB : -1; }
    // Loads that a wave issues between the load a wait is for and the wait, the
    // least over the first bodies and the steady state: 'a' the activation
    // stage met at unit us, 'b' the weight stage first read in unit us, 'w'
    // the next body's w_s; 's' the loop's start, where the first stage of each
    // (and as many activations as the first fragments reach) have landed.
    static constexpr int behind(char what, int us) {
        int least = 1 << 30;
        for (int body = 0; body < 6; ++body) {
            int n = 0, at = -1;
            const int end = 4 * body + us;  // the wait's unit
            for (int u = -8; u <= end; ++u) {
                if (what == 's' && u == 0) break;
                if (what == 'a' && u == end) break;
                if (a_stage(u) >= 0) {
                    n += NA + 1;
                    if (what == 'a' ? a_stage(u) == end / SU + 1 : what == 's' && a_stage(u) <= (PD - 1) / (A * SU)) at = n;
                }
                if (what == 'b' && u == end) break;
                if (w_body(u) >= 0) {
                    n += B * WST;
                    if (what == 'w' ? w_body(u) == body + 1 : what == 's' && w_body(u) == 0) at = n;
                }
                if (b_stage(u) >= 0 && !(what == 's' && b_stage(u) >= NB)) {
                    n += 2 * B;
                    if (what == 'b' ? b_stage(u) == (end + 1) / UB : what == 's' && b_stage(u) == 0) at = n;
                }
            }
            least = at < 0 ? -1 : n - at < least ? n - at : least;
            if (at < 0) break;
        }
        return least;
    }
    static constexpr bool waits() {  // every wait's load is among those before it
        for (int us = 0; us < 4; ++us)
            if ((a_stage(us) >= 0 && behind('a', us) < 0) || ((us + 1) % UB == 0 && behind('b', us) < 0)) return false;
        return behind('w', 3) >= 0 && behind('s', 0) >= 0;
    }
};

template <typename T, int MINB, bool HQ>
__global__ __launch_bounds__(64 * T::NW, MINB) void gemm_t16_kernel(
    const unsigned char *Af, const float *asf, const int8_t *W0, const float *S0, int Mt, int N,
    int K, int M, const int8_t *W1, GemmT16Args args) {
    constexpr int GS = T::GS, A = T::A, B = T::B, NW = T::NW, SU = T::SU, NB = T::NB, NT = T::NT, NJ = T::NJ;
    constexpr int COLS = T::COLS, MT = T::MT, UC = T::UC, GU = T::GU, UB = T::UB, NM = T::NM, SC = T::SC;
    constexpr int SG = T::SG, NG = T::NG, PD = T::PD, CB = T::CB, ABUF = T::ABUF, SBUF = T::SBUF, WST = T::WST;
    constexpr int NAS = (A + 3) / 4;  // scale registers of a group (64 rows each)
    constexpr bool SWIGLU = T::SWIGLU;
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, nl = lane & 15;
    const int Kc = K / 64, Kg = K / GS;
    // XCD-aware tile order. Workgroups go to the 8 XCDs round-robin (block b
    // to XCD b % 8), and each XCD has its own L2: XCD x takes the contiguous
    // tiles [x per, (x+1) per), M-tile fastest, so a few columns of weight
    // rows meet all activation rows in one L2.
    const int tiles_m = (Mt + MT - 1) / MT;
    const int tiles = tiles_m * ((N + COLS - 1) / COLS);
    const int per = (tiles + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= tiles || (int)(blockIdx.x / 8) >= per) return;  // whole block: before any barrier
    const int n0 = (t / tiles_m) * COLS, mt0 = (t % tiles_m) * MT;

    // Buffer resources based at the block's own rows; the advance along K
    // goes in the scalar offset.
    const int mtn = min(MT, Mt - mt0), rows = N - n0;
    const rsrc_t rA = make_rsrc(Af + (size_t)mt0 * Kc * 4096, (uint32_t)mtn * Kc * 4096);
    const rsrc_t rAS = make_rsrc(asf + (size_t)mt0 * Kg * 32, (uint32_t)mtn * Kg * 128);
    const rsrc_t rW0 = make_rsrc(W0 + (size_t)n0 * K, (uint32_t)rows * K);
    const rsrc_t rW1 = make_rsrc((SWIGLU ? W1 : W0) + (size_t)n0 * K, (uint32_t)rows * K);
    const rsrc_t rS0 = make_rsrc(S0 + (size_t)n0 * Kg, (uint32_t)rows * Kg * 4);
    const rsrc_t rS1 = make_rsrc((SWIGLU ? args.S1 : S0) + (size_t)n0 * Kg, (uint32_t)rows * Kg * 4);

    // ---- activations: the waves copy a stage's fragments and scales linearly
    // in 1 KB pieces (m-tiles past the product are clamped; the scales' pieces
    // repeat over the waves, the same bytes to the same place)
    int aoff[T::NA], asoff;
#pragma unroll
    for (int i = 0; i < T::NA; ++i) {
        const int p = wid + NW * i, mt = p / (SC * 4);
        aoff[i] = min(mt, mtn - 1) * Kc * 4096 + (p % (SC * 4)) * 1024 + lane * 16;
    }
    const int spiece = wid % (SBUF / 1024);
    {
        const int o = min(spiece * 1024 + lane * 16, T::SBYTES - 16), mt = o / (SG * 128);
        asoff = min(mt, mtn - 1) * Kg * 128 + o % (SG * 128);
    }
    // ---- weights: a stage takes 128 bytes of each of a tile's 16 rows, 8 rows
    // a load: 8 consecutive lanes read one row's 128 bytes (16 lanes spread
    // over 16 rows, the order the MFMA wants, cost six times as much in the
    // vector cache). LDS slot 8 row + s holds the row's 16-byte piece s ^
    // ((row / 2) & 7), so that a fragment read meets 16 different bank groups.
    // w_s: four groups of each row, 4 lanes a row.
    int woff[B][2], soff[B];
#pragma unroll
    for (int j = 0; j < B; ++j) {
        const int r0 = 16 * (wid * NJ + j % NJ);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = 8 * i + (lane >> 3);
            woff[j][i] = min(r0 + r, rows - 1) * K + 16 * ((lane & 7) ^ ((r >> 1) & 7));
        }
        soff[j] = (min(r0 + (lane >> 2), rows - 1) * Kg + (lane & 3)) * 4;
    }
    const int bbase = T::OFF_B + wid * B * NB * 2048, wbase = T::OFF_W + wid * 2 * B * WST * 256;
    auto load_a = [&](int buf, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < T::NA; ++i) dma16(rA, aoff[i], stage * SC * 4096, buf * ABUF + (wid + NW * i) * 1024);
        dma16(rAS, asoff, stage * SG * 128, T::OFF_S + buf * SBUF + spiece * 1024);
    };
    auto load_b = [&](int sl, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < B; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                dma16(SWIGLU && j >= NJ ? rW1 : rW0, woff[j][i], stage * 128, bbase + (j * NB + sl) * 2048 + i * 1024);
    };
    auto load_ws = [&](int sl, int body) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < B; ++j)
#pragma unroll
            for (int h = 0; h < WST; ++h)
                dma4(SWIGLU && j >= NJ ? rS1 : rS0, soff[j], (body * NG + 4 * h) * 4, wbase + ((sl * B + j) * WST + h) * 256);
    };

    float4_t out[A][B];
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) out[i][j] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};

    // this lane's place in a group's scales of a 64-row range: DPP row r's 16
    // lanes hold what rows 16 i + 4r + e need, in lane 4 i + e
    const int asl = (A >= 4 ? ((lane >> 3) & 1) * SG * 32 : 0) + (lane >> 4) * 8 + (lane & 7);
    const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    half8_t fr[4][NM];                 // activation fragments of four steps
    float4_t acc[2][B][GU];            // group sums of two steps
    u32x4 raw[B][UC];                  // the next unit's weights
    uint32_t bf[2][B][NM][4];          // widened weights of two units
    float as[2][GU][NAS];              // scales of two units
    float wsn[B][NG];                  // the next body's w_s
    // fragments of row tile i / the scales of unit u of the stage in buffer buf
    auto read_fr = [&](int sl, int buf, int u, int i) __attribute__((always_inline)) {
        const u32x4 *p = reinterpret_cast<const u32x4 *>(smem + buf * ABUF) + ((i >> 1) * SC + u * UC) * 256 + (i & 1) * 128 + lane;
#pragma unroll
        for (int k = 0; k < NM; ++k) fr[sl][k] = __builtin_bit_cast(half8_t, p[(k >> 1) * 256 + (k & 1) * 64]);
    };
    auto read_as = [&](int sl, int buf, int u) __attribute__((always_inline)) {
        const float *p = reinterpret_cast<const float *>(smem + T::OFF_S + buf * SBUF);
#pragma unroll
        for (int g = 0; g < GU; ++g)
#pragma unroll
            for (int n = 0; n < NAS; ++n) as[sl][g][n] = p[n * 2 * SG * 32 + (u * GU + g) * 32 + asl];
    };
    // this lane's weights of unit u of the stage in slot sl
    auto read_raw = [&](int sl, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const unsigned char *p = smem + bbase + (j * NB + sl) * 2048 + nl * 128;
#pragma unroll
            for (int x = 0; x < UC; ++x) {
                if constexpr (GS == 32) {  // 8 bytes of each of the chunk's two groups
                    const u32x2 g0 = *reinterpret_cast<const u32x2 *>(p + (((4 * u + (c >> 1)) ^ (nl >> 1)) & 7) * 16 + 8 * (c & 1));
                    const u32x2 g1 = *reinterpret_cast<const u32x2 *>(p + (((4 * u + 2 + (c >> 1)) ^ (nl >> 1)) & 7) * 16 + 8 * (c & 1));
                    raw[j][x] = (u32x4){g0[0], g0[1], g1[0], g1[1]};
                } else {
                    raw[j][x] = *reinterpret_cast<const u32x4 *>(p + (((4 * (u * UC + x) + c) ^ (nl >> 1)) & 7) * 16);
                }
            }
        }
    };
    auto read_ws = [&](int sl) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < B; ++j)
#pragma unroll
            for (int h = 0; h < WST; ++h) {
                const float4 v = *reinterpret_cast<const float4 *>(smem + wbase + ((sl * B + j) * WST + h) * 256 + nl * 16);
                wsn[j][4 * h] = v.x;
                wsn[j][4 * h + 1] = v.y;
                wsn[j][4 * h + 2] = v.z;
                wsn[j][4 * h + 3] = v.w;
            }
    };
    // MFMA k of a step's tiles
    auto mfma = [&](int fs, int sl, int bs, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const half8_t b = __builtin_bit_cast(half8_t, (u32x4){bf[bs][j][k][0], bf[bs][j][k][1], bf[bs][j][k][2], bf[bs][j][k][3]});
            const int g = GU == 2 ? k : 0;
            acc[sl][j][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fr[fs][k], b, (GU == 2 || k == 0) ? zero : acc[sl][j][g], 0, 0, 0);
        }
    };
    // out = fma(G * a_s, w_s, out) (reference order): the product first, a_s
    // coming by DPP row broadcast, the sum in a second pass over the same
    // elements (each product has its own register: one reused right away
    // would wait out a hazard)
    auto scale1 = [&](float a_s, float g, int ctrl) __attribute__((always_inline)) {
        const int v = __builtin_bit_cast(int, a_s);
        int b = 0;
        switch (ctrl) {  // (an immediate operand)
#define Q3VL_C(X) case X: b = __builtin_amdgcn_mov_dpp(v, 0x150 + X, 0xF, 0xF, true); break;
            Q3VL_C(0) Q3VL_C(1) Q3VL_C(2) Q3VL_C(3) Q3VL_C(4) Q3VL_C(5) Q3VL_C(6) Q3VL_C(7)
            Q3VL_C(8) Q3VL_C(9) Q3VL_C(10) Q3VL_C(11) Q3VL_C(12) Q3VL_C(13) Q3VL_C(14) Q3VL_C(15)
#undef Q3VL_C
        }
        return __builtin_bit_cast(float, b) * g;
    };
    // part k of NM of the folds of step i (us: the unit's place in the body;
    // sums in acc[sl]): elements x of group g, tile x / 4
    constexpr int FE = GU == 2 ? 4 * B : 4 * B / NM;
    auto scale = [&](int i, int us, int sl, int k, float (&tt)[FE]) __attribute__((always_inline)) {
        const int g = GU == 2 ? k : 0, x0 = GU == 2 ? 0 : k * FE;
#pragma unroll
        for (int y = 0; y < FE; ++y)
            tt[y] = scale1(as[us & 1][g][i / 4], acc[sl][(x0 + y) / 4][g][(x0 + y) % 4], 4 * (i % 4) + (x0 + y) % 4);
    };
    auto fold = [&](int i, int us, int k, const float (&tt)[FE], const float (&ws)[B][NG]) __attribute__((always_inline)) {
        const int g = GU == 2 ? k : 0, x0 = GU == 2 ? 0 : k * FE;
#pragma unroll
        for (int y = 0; y < FE; ++y)
            out[i][(x0 + y) / 4][(x0 + y) % 4] = fmaf(tt[y], ws[(x0 + y) / 4][us * GU + g], out[i][(x0 + y) / 4][(x0 + y) % 4]);
    };
    // dword d of B * UC * 4 of raw, widened into bf[bs]
    auto widen = [&](int bs, int d) __attribute__((always_inline)) {
        const int j = d / (UC * 4), u = d / 4 % UC, w = d % 4;
        widen4(raw[j][u][w], bf[bs][j][2 * u + w / 2][2 * (w & 1)], bf[bs][j][2 * u + w / 2][2 * (w & 1) + 1]);
    };
    constexpr int ND = B * UC * 4;           // dwords to widen per unit
    constexpr int NSUB = (A - 1) * NM;       // sub-steps that widen (the next unit's first MFMA follows)

    const int nbody = Kc / (4 * UC), last = 4 * nbody - 1, lasta = last / SU, lastb = last / UB;
    int b0 = 0, b1 = 1, b2 = 2;  // activation buffers of this, the next and the stage after
    int sb = 0;                  // weight slot of the stage that holds the next unit
    // One unit n (us: its place among the four of the loop body). On entry its
    // weights are widened in bf[us & 1], its scales read, the fragments of
    // steps 0 .. PD-1 read and step 0's MFMAs issued.
    auto unit = [&](auto usc, int n, const float (&ws)[B][NG]) __attribute__((always_inline)) {
        constexpr int us = decltype(usc)::value, su = us % SU;
        if constexpr (su == SU - CB) {
            // the next stage has landed for every wave, and every wave is past
            // the previous one, whose buffer the stage after the next takes
            dma_wait<T::behind('a', us)>();
            lds_barrier();
            load_a(b2, min(n / SU + 2, lasta));
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr ((us + 1) % UB == 0) dma_wait<T::behind('b', us)>();
        read_raw(sb, (us + 1) % UB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < A; ++i) {
            // fragments PD steps ahead, MFMAs one step ahead, folds of this one
            const int st = us * A + i, ru = su + (i + PD) / A;
            if (i == A - 1) read_as((us + 1) & 1, su == SU - 1 ? b1 : b0, (su + 1) % SU);
            read_fr((st + PD) & 3, ru >= SU ? (ru >= 2 * SU ? b2 : b1) : b0, ru % SU, (i + PD) % A);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                float tt[FE];
                mfma((st + 1) & 3, (i + 1) & 1, i + 1 < A ? us & 1 : (us + 1) & 1, k);
                __builtin_amdgcn_sched_barrier(0);
                scale(i, us, i & 1, k, tt);
                __builtin_amdgcn_sched_barrier(0);
                if (i + 1 < A) {
                    const int sub = i * NM + k;
#pragma unroll
                    for (int x = 0; x < ND; ++x)
                        if (x * NSUB / ND == sub) widen((us + 1) & 1, x);
                }
                __builtin_amdgcn_sched_barrier(0);
                fold(i, us, k, tt, ws);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (us == 0 && i == 0) {
                // this body's w_s (read at the last one's end) are in their
                // registers: before that their slot must not be refilled, and
                // nothing else orders the refill behind the reads. By now the
                // wait costs nothing; at the unit's start it would.
#pragma unroll
                for (int j = 0; j < B; ++j)
#pragma unroll
                    for (int k = 0; k < NG; ++k) asm volatile("" ::"v"(ws[j][k]));
                load_ws((n >> 2) & 1, min((n >> 2) + 2, nbody - 1));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (i + 2 == A && (us + 1) % UB == UB - 1) {  // the slot is consumed
                load_b(sb, min((n + 1) / UB + NB, lastb));
                sb = sb + 1 == NB ? 0 : sb + 1;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (us == 3) {
            dma_wait<T::behind('w', 3)>();
            read_ws(((n >> 2) + 1) & 1);
        }
        if constexpr (su == SU - 1) {
            const int x = b0;
            b0 = b1;
            b1 = b2;
            b2 = x;
        }
    };
    static_assert(2 * SU > SU - 1 + (A - 1 + PD) / A, "fragments are read at most one stage ahead");

    if (nbody > 0) {
        static_assert(T::waits(), "loads");
#pragma unroll
        for (int u = -8; u < 0; ++u) {  // (slot: the stage's number; one past the slots goes out below)
            if (T::a_stage(u) >= 0) load_a(T::a_stage(u), min(T::a_stage(u), lasta));
            if (T::w_body(u) >= 0) load_ws(T::w_body(u), min(T::w_body(u), nbody - 1));
            if (T::b_stage(u) >= 0 && T::b_stage(u) < NB) load_b(T::b_stage(u), min(T::b_stage(u), lastb));
        }
        dma_wait<T::behind('s', 0)>();
        lds_barrier();
        read_ws(0);
        read_as(0, 0, 0);
#pragma unroll
        for (int x = 0; x < PD; ++x) read_fr(x, x / A >= SU ? 1 : 0, x / A % SU, x % A);
        read_raw(0, 0);
#pragma unroll
        for (int x = 0; x < ND; ++x) widen(0, x);
        if (UB == 1) {
            __builtin_amdgcn_sched_barrier(0);
            load_b(0, min(NB, lastb));
            sb = 1;
        }
#pragma unroll
        for (int k = 0; k < NM; ++k) mfma(0, 0, 0, k);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int q = 0; q < nbody; ++q) {
        float ws[B][NG];
#pragma unroll
        for (int j = 0; j < B; ++j)
#pragma unroll
            for (int k = 0; k < NG; ++k) ws[j][k] = wsn[j][k];
        unit(std::integral_constant<int, 0>{}, 4 * q, ws);
        unit(std::integral_constant<int, 1>{}, 4 * q + 1, ws);
        unit(std::integral_constant<int, 2>{}, 4 * q + 2, ws);
        unit(std::integral_constant<int, 3>{}, 4 * q + 3, ws);
    }
    dma_wait<0>();  // (the loads past the last unit)
    // units past the whole bodies (K not a multiple of 256 UC): one at a time
    const int u0 = 4 * nbody, nu = Kc / UC;
    for (int n = u0; n < nu; ++n) {
        lds_barrier();  // the buffer is free
        for (int p = tid; p < MT * UC * 256; p += NT) {
            const int mt = p / (UC * 256), r = p % (UC * 256);
            *reinterpret_cast<u32x4 *>(smem + (mt * SC * 256 + r) * 16) = *reinterpret_cast<const u32x4 *>(
                Af + ((size_t)(mt0 + min(mt, mtn - 1)) * Kc + n * UC) * 4096 + r * 16);
        }
        for (int p = tid; p < MT * GU * 32; p += NT) {
            const int mt = p / (GU * 32), r = p % (GU * 32);
            reinterpret_cast<float *>(smem + T::OFF_S)[mt * SG * 32 + r] =
                asf[((size_t)(mt0 + min(mt, mtn - 1)) * Kg + n * GU) * 32 + r];
        }
        float ws[B][NG];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int row = n0 + min(16 * (wid * NJ + j % NJ) + nl, rows - 1);
            const int8_t *w = (SWIGLU && j >= NJ ? W1 : W0) + (size_t)row * K + (size_t)n * UC * 64;
            const float *s = (SWIGLU && j >= NJ ? args.S1 : S0) + (size_t)row * Kg + n * GU;
#pragma unroll
            for (int k = 0; k < GU; ++k) ws[j][k] = s[k];
#pragma unroll
            for (int x = 0; x < UC; ++x) {
                if constexpr (GS == 32) {
                    const u32x2 g0 = *reinterpret_cast<const u32x2 *>(w + 8 * c), g1 = *reinterpret_cast<const u32x2 *>(w + 32 + 8 * c);
                    raw[j][x] = (u32x4){g0[0], g0[1], g1[0], g1[1]};
                } else {
                    raw[j][x] = *reinterpret_cast<const u32x4 *>(w + 64 * x + 16 * c);
                }
            }
        }
        lds_barrier();
        read_as(0, 0, 0);
#pragma unroll
        for (int x = 0; x < ND; ++x) widen(0, x);
#pragma unroll
        for (int i = 0; i < A; ++i) {
            read_fr(0, 0, 0, i);
#pragma unroll
            for (int k = 0; k < NM; ++k) mfma(0, 0, 0, k);
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                float tt[FE];
                scale(i, 0, 0, k, tt);
                fold(i, 0, k, tt, ws);
            }
        }
    }
    lds_barrier();

    // ---- SwiGLU with hq: the block's h tile (16 A rows x COLS columns, whole
    // groups of the down projection's K) quantized straight into the down
    // GEMM's operand in place of storing h. Rows past M get q = 0 and a_s = 0,
    // as the quantizer's padding rows do.
    if constexpr (SWIGLU && HQ) {
        constexpr int HLD = COLS + 4;
        static_assert(COLS % GS == 0, "whole groups");
        float *ht = reinterpret_cast<float *>(smem);  // (the last barrier has passed)
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float gv[4] = {out[i][j][0], out[i][j][1], out[i][j][2], out[i][j][3]};
                const float uv[4] = {out[i][j + NJ][0], out[i][j + NJ][1], out[i][j + NJ][2], out[i][j + NJ][3]};
                float h[4];
                silu_mul_n<4>(gv, uv, h);
#pragma unroll
                for (int e = 0; e < 4; ++e) ht[(16 * i + 4 * c + e) * HLD + 16 * (wid * NJ + j) + nl] = h[e];
            }
        lds_barrier();
        constexpr int GB = COLS / GS;  // groups of the tile
        for (int p = tid; p < 16 * A * GB * 4; p += NT) {
            const int j = p & 3, g = (p >> 2) % GB, rr = (p >> 2) / GB;
            const int mt = mt0 + (rr >> 5), r = rr & 31;
            const bool real = 32 * mt + r < M;
            float4 cv[GS / 16];
#pragma unroll
            for (int v = 0; v < GS / 16; ++v)
                cv[v] = real ? *reinterpret_cast<const float4 *>(ht + rr * HLD + g * GS + 16 * v + 4 * j)
                             : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const bool in = mt < Mt && n0 + g * GS < N;  // (a block's last tiles may lie past the product)
            const float s = quant_team<GS>(cv, [&](int v, uint32_t h0, uint32_t h1) {
                if (in)
                    *reinterpret_cast<uint2 *>(reinterpret_cast<unsigned char *>(args.hq) +
                                               frag_off<GS>(mt, r, N / 64, n0 + g * GS + 16 * v + 4 * j)) =
                        real ? make_uint2(h0, h1) : make_uint2(0u, 0u);
            });
            if (in && j == 0) args.hqs[frag_scale(mt, r, N / GS, n0 / GS + g)] = real ? s : 0.0f;
        }
        return;
    }

    // ---- greedy-argmax partials of the block's columns (plain products): per
    // row the larger value, equal values the lower column, values that are
    // not above -FLT_MAX never win -- the strict > scan from -FLT_MAX. Each
    // lane reduces its B columns (the others hold -FLT_MAX), the 16 lanes of a
    // row group take the largest value and then the lowest column that has it
    // by DPP, the waves meet in LDS (free: the last barrier has passed). As xor
    // shuffles through LDS, value and column together, this took about 15 us a
    // round of 128 x 128 blocks: lm_head [151936, 2048] at 65 rows 211 us,
    // now 166.
    if constexpr (!SWIGLU) {
        if (args.part_val) {  // uniform
            float *rv = reinterpret_cast<float *>(smem);  // [NW][16 A]
            int32_t *ri = reinterpret_cast<int32_t *>(rv + NW * 16 * A);
#pragma unroll
            for (int i = 0; i < A; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float bv = -FLT_MAX;
                    int32_t bi = -1;
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        const int col = n0 + 16 * (wid * B + j) + nl;
                        if (col < N && out[i][j][e] > -FLT_MAX) am_combine(bv, bi, out[i][j][e], col);
                    }
                    const float top = row16_max(bv);
                    bi = row16_min(bv == top && bi >= 0 ? bi : INT_MAX);
                    bv = top;
                    if (bi == INT_MAX) bi = -1;
                    if (nl == 0) {
                        rv[wid * 16 * A + 16 * i + 4 * c + e] = bv;
                        ri[wid * 16 * A + 16 * i + 4 * c + e] = bi;
                    }
                }
            lds_barrier();
            for (int r = tid; r < 16 * A; r += NT) {
                float bv = -FLT_MAX;
                int32_t bi = -1;
#pragma unroll
                for (int w = 0; w < NW; ++w) am_combine(bv, bi, rv[w * 16 * A + r], ri[w * 16 * A + r]);
                const int mrow = 32 * mt0 + r;
                if (mrow < M) {
                    args.part_val[(size_t)(n0 / COLS) * M + mrow] = bv;
                    args.part_idx[(size_t)(n0 / COLS) * M + mrow] = bi;
                }
            }
        }
    }

    // ---- store (an argmax caller that wants no logits passes C = null)
    if (!args.C) return;  // uniform
    if constexpr (SWIGLU) {
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float gv[4] = {out[i][j][0], out[i][j][1], out[i][j][2], out[i][j][3]};
                const float uv[4] = {out[i][j + NJ][0], out[i][j + NJ][1], out[i][j + NJ][2], out[i][j + NJ][3]};
                float h[4];
                silu_mul_n<4>(gv, uv, h);
#pragma unroll
                for (int e = 0; e < 4; ++e) out[i][j][e] = h[e];
            }
    }
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int mrow = 32 * mt0 + 16 * i + 4 * c + e;
            if (mrow >= M) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int col = n0 + 16 * (wid * NJ + j) + nl;
                if (col < N)
                    args.C[(size_t)mrow * N + col] = out[i][j][e];
            }
        }
}

template <typename T, int MINB, bool HQ = false>
static hipError_t launch_t16(const GemmT16Args &a, hipStream_t st) {
    const int tiles = ((a.N + T::COLS - 1) / T::COLS) * ((a.Mt + T::MT - 1) / T::MT);
    const int grid = 8 * ((tiles + 7) / 8);
    constexpr int htile = HQ ? 16 * T::A * (T::COLS + 4) * 4 : 0;
    constexpr int am = T::SWIGLU ? 0 : T::NW * 16 * T::A * 8;
    constexpr int lds = T::LDS > htile ? (T::LDS > am ? T::LDS : am) : htile;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_t16_kernel<T, MINB, HQ>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    gemm_t16_kernel<T, MINB, HQ><<<grid, 64 * T::NW, lds, st>>>(reinterpret_cast<const unsigned char *>(a.Af), a.asf, a.W0,
                                                               a.S0, a.Mt, a.N, a.K, a.M, a.W1, a);
    return hipGetLastError();
}

// Which tile. A tile's blocks run in rounds of `cap` blocks a CU; a round of
// L blocks a CU takes fix + unit[L - 1] * K / 64 us, and tail us for each unit
// of K past the whole loop bodies, which run one at a time (0.3 to 1 us each
// on top: 65 x 12288 at K = 256 / 384 / 512 takes 10.5 / 13.9 / 12.3 us in
// tiles of 32 x 128). The plain tables are fitted to the tiles' times, each
// forced, over 4500 products at groups 32 and 64 and 2200 at 128 (M 17 to
// 2048, N 512 to 50000, K 128 to 6144, cold caches): the tile taken is 0.3 %
// (0.5 % at group 128) slower than the best one on average, 22 % at most; with
// tables read off a few large products, and no tail, it was 1.7 % and 59 %,
// most of it at K up to 512 (65 x 50000 x 384 32 us, 20.6 in the best tile).
// The product takes the tile whose rounds cost least. Small products want one small block on every CU, larger
// ones two or three blocks of 64 x 64, which wait at barriers of their own
// (4 waves each), and where those leave a round half empty, larger blocks:
// * plain (us; 32 x 64 / 32 x 128 / 64 x 64 / 64 x 128 / 128 x 128):
//     196 x 2048 x 4096   14.7 /  -   /  -   /  -   /  -
//     512 x 2048 x 6144   30.5 / 26.9 / 39.6 / 43.5 / 63
//     784 x 3072 x 1024   17.3 / 18.2 / 13.6 / 15.5 / 15.9
//     784 x 4096 x 1024    -   /  -   / 18.0 / 16.3 / 16.6
//     1000 x 2048 x 6144  65.5 / 54.9 / 46.3 / 48.0 / 65.6
//     1501 x 2048 x 6144   -   /  -   / 66.8 / 71.4 / 69.4
//     1501 x 4096 x 2048   -   /  -   / 47.1 / 44.1 / 52.8
//   and at group 128 1501 x 2048 x 6144 68 / 71 / 58 (64 x 64, 64 x 128, 128 x 128);
// * SwiGLU (output columns, each a gate and an up column; 32 x 64 / 64 x 64 /
//   128 x 128), N = 6144, K = 2048: 16 rows 12.7 / 19.7 / 41.7, 200 rows 28.0
//   / 27.5 / 43.2, 300 rows 36.3 / 28.8 / -, 512 rows - / 45.8 / 48.3, 1501
//   rows 166 / 130 / 131. Up to one block a CU the 32 x 64 tile takes longer
//   stages of activations (12.7 us, 13.3 without). At group 128 a tile has
//   128 columns (whole groups of the h it quantizes) and at most 64 rows
//   (more spill): 300 rows 31 (32 x 128), 26 (64 x 128).
// A large product's last round is often nearly empty (1501 x 6144 SwiGLU: 576
// blocks of 128 x 128, 2.25 rounds): the rows of the whole rounds then run
// first, and the rest as a product of its own, with its own tile, where the
// two and another launch cost less (at 1501 rows 88 us + 27 in place of 130).
struct T16Tile {
    int rows, cols, cap;
    float unit[3], fix, tail;
};
struct T16Plan {
    int tile, rows, tile2;  // rows 0 .. rows - 1 by tile, the others (if any) by tile2
};
enum { P32x64, P32x128, P64x64, P64x128, P128x128, PLAIN_TILES };
static const T16Tile kPlain[PLAIN_TILES] = {{32, 64, 1, {0.20f}, 2.5f, 0.3f},
                                            {32, 128, 1, {0.33f}, 2.5f, 0.55f},
                                            {64, 64, 3, {0.36f, 0.38f, 0.61f}, 5.2f, 0.7f},
                                            {64, 128, 2, {0.39f, 0.67f}, 5.3f, 0.48f},
                                            {128, 128, 1, {0.66f}, 5.7f, 0.97f}};
static const T16Tile kPlain128[PLAIN_TILES] = {{32, 64, 1, {0.21f}, 3.1f, 0.52f},
                                               {32, 128, 1, {0.31f}, 2.3f, 0.55f},
                                               {64, 64, 3, {0.32f, 0.40f, 0.68f}, 9.4f, 0.92f},
                                               {64, 128, 2, {0.33f, 0.91f}, 5.9f, 0.56f},
                                               {128, 128, 1, {0.54f}, 4.7f, 0.73f}};
enum { S32x64L, S32x64, S64x64, S128x128, SWIGLU_TILES };
static const T16Tile kSwiglu[SWIGLU_TILES] = {{32, 64, 1, {0.18f}, 7, 0},
                                              {32, 64, 2, {0.20f, 0.36f}, 7, 0},
                                              {64, 64, 2, {0.35f, 0.61f}, 7.5f, 0},
                                              {128, 128, 1, {1.16f}, 9, 0}};
enum { S32x128, S64x128, SWIGLU128_TILES };
static const T16Tile kSwiglu128[SWIGLU128_TILES] = {{32, 128, 1, {0.25f}, 8, 0}, {64, 128, 1, {0.55f}, 8, 0}};

static T16Plan t16_plan(int M, int N, int K, int gs, bool swiglu, bool argmax, int cus) {
    const T16Tile *tiles = swiglu ? (gs == 128 ? kSwiglu128 : kSwiglu) : gs == 128 ? kPlain128 : kPlain;
    const int n = swiglu ? (gs == 128 ? (int)SWIGLU128_TILES : (int)SWIGLU_TILES) : (int)PLAIN_TILES;
    const float units = (float)K / 64, tail = (float)(K / (gs == 128 ? 128 : 64) % 4);
    auto cost = [&](const T16Tile &q, int m) {
        // (64 rows for at most 32 are half padding: faster for their epilogue
        // at a small K alone, 24 x 50000 x 128 13 % so; 16 x 50000 x 4224 at group
        // 32 takes 79 us in 64 x 128 tiles, 69 in 32 x 128)
        if (!swiglu && m <= 32 && q.rows > 32 && K >= 1024) return 1e30f;
        const long blocks = (long)((m + q.rows - 1) / q.rows) * ((N + q.cols - 1) / q.cols);
        const long slots = (long)q.cap * cus, rounds = (blocks - 1) / slots;
        const long level = (blocks - rounds * slots - 1) / cus;  // of the last round
        return (float)rounds * (q.fix + q.unit[q.cap - 1] * units + q.tail * tail) + q.fix + q.unit[level] * units +
               q.tail * tail;
    };
    T16Plan best{0, M, 0};
    float least = 1e30f;
    for (int t = 0; t < n; ++t) {
        // (the 64-column tiles leave twice the argmax partials: only where
        // they are few)
        if (argmax && tiles[t].cols == 64 && (long)((M + 31) / 32) * ((N + 63) / 64) > cus) continue;
        const float c = cost(tiles[t], M);
        if (c < least) {
            least = c;
            best = {t, M, 0};
        }
    }
    if (argmax) return best;  // (one set of partials)
    const T16Tile &big = tiles[n - 1];
    const long nb = (N + big.cols - 1) / big.cols;
    for (int r = 1; r <= 16; ++r) {  // r whole rounds of the largest tile
        const long m1 = (long)r * cus / nb * big.rows;
        if (m1 >= M) break;
        if (m1 <= 0) continue;
        const float c1 = cost(big, (int)m1) + 2;
        for (int t = 0; t < n; ++t) {
            const float c = c1 + cost(tiles[t], M - (int)m1);
            if (c < least) {
                least = c;
                best = {n - 1, (int)m1, t};
            }
        }
    }
    return best;
}

void gemm_t16_tiles(int M, int N, int K, int gs, bool swiglu, bool argmax, int cus, int out[3]) {
    const T16Plan p = t16_plan(M, N, K, gs, swiglu, argmax, cus);
    out[0] = p.tile;
    out[1] = p.rows;
    out[2] = p.tile2;
}

// Columns per argmax partial of a plain product.
int gemm_t16_argmax_cols(int M, int N, int K, int gs, int cus) {
    return kPlain[t16_plan(M, N, K, gs, false, true, cus).tile].cols;  // (the same at every group size)
}

// The kernel addresses a block's rows with 32-bit byte offsets.
bool gemm_t16_serves(int M, int N, int K, int gs) {
    return (gs == 32 || gs == 64 || gs == 128) && K > 0 && K % 64 == 0 && K % gs == 0 && K <= (1 << 22) && M >= 1 &&
           N >= 1;
}

template <int GS> static hipError_t launch_plain(const GemmT16Args &a, int tile, hipStream_t st) {
    constexpr int S4 = GS == 128 ? 2 : 4;  // a stage of 256 k (the loads of more do not fit the counter)
    // (four waves: two blocks' worth of registers, or the sums would move
    // through accumulation registers, 16.5 us instead of 14.7 at 196 x 2048 x 4096)
    if (tile == P32x64) return launch_t16<T16<GS, 2, 1, 4, S4, 3, false>, 2>(a, st);
    if (tile == P32x128) return launch_t16<T16<GS, 2, 1, 8, S4, 2, false>, 1>(a, st);
    if (tile == P64x64) return launch_t16<T16<GS, 4, 1, 4, 1, 2, false>, 3>(a, st);
    if (tile == P64x128) return launch_t16<T16<GS, 4, 1, 8, 1, 2, false>, 2>(a, st);
    return launch_t16<T16<GS, 8, 1, 8, 1, 2, false>, 1>(a, st);
}

template <int GS, bool HQ> static hipError_t launch_swiglu(const GemmT16Args &a, int tile, hipStream_t st) {
    if constexpr (GS == 128) {
        if (tile == S32x128) return launch_t16<T16<GS, 2, 2, 8, 2, 2, true>, 1, HQ>(a, st);
        return launch_t16<T16<GS, 4, 2, 8, 1, 2, true>, 1, HQ>(a, st);
    } else {
        if (tile == S32x64L) return launch_t16<T16<GS, 2, 2, 4, 4, 2, true>, 2, HQ>(a, st);
        if (tile == S32x64) return launch_t16<T16<GS, 2, 2, 4, 2, 2, true>, 2, HQ>(a, st);
        if (tile == S64x64) return launch_t16<T16<GS, 4, 2, 4, 1, 2, true>, 2, HQ>(a, st);
        return launch_t16<T16<GS, 8, 2, 8, 1, 2, true>, 1, HQ>(a, st);
    }
}

template <int GS> static hipError_t launch_tile(const GemmT16Args &a, bool swiglu, int tile, hipStream_t st) {
    if (!swiglu) return launch_plain<GS>(a, tile, st);
    return a.hq ? launch_swiglu<GS, true>(a, tile, st) : launch_swiglu<GS, false>(a, tile, st);
}

template <int GS> static hipError_t launch_gs(const GemmT16Args &a, bool swiglu, int cus, hipStream_t st) {
    const T16Plan p = t16_plan(a.M, a.N, a.K, GS, swiglu, a.part_val != nullptr, cus);
    if (p.rows >= a.M) return launch_tile<GS>(a, swiglu, p.tile, st);
    GemmT16Args x = a, y = a;  // (p.rows: whole 32-row m-tiles)
    x.M = p.rows;
    x.Mt = p.rows / 32;
    y.M = a.M - p.rows;
    y.Mt = a.Mt - x.Mt;
    y.Af += (size_t)p.rows * a.K;
    y.asf += (size_t)p.rows * (a.K / GS);
    if (a.C) y.C += (size_t)p.rows * a.N;
    if (a.hq) {
        y.hq += (size_t)p.rows * a.N;
        y.hqs += (size_t)p.rows * (a.N / GS);
    }
    const hipError_t e = launch_tile<GS>(x, swiglu, p.tile, st);
    return e != hipSuccess ? e : launch_tile<GS>(y, swiglu, p.tile2, st);
}

hipError_t launch_gemm_t16(const GemmT16Args &a, int gs, bool swiglu, int cus, hipStream_t st) {
    if (!gemm_t16_serves(a.M, a.N, a.K, gs) || a.Mt != (a.M + 31) / 32) return hipErrorInvalidValue;
    if (swiglu && a.part_val) return hipErrorInvalidValue;
    // h quantized in the epilogue: SwiGLU only, whole groups and chunks
    if (a.hq && (!swiglu || !a.hqs || a.N % 64 != 0 || a.N % gs != 0)) return hipErrorInvalidValue;
    if (gs == 32) return launch_gs<32>(a, swiglu, cus, st);
    if (gs == 64) return launch_gs<64>(a, swiglu, cus, st);
    return launch_gs<128>(a, swiglu, cus, st);
}

}  // namespace q3vl
