// The GEMM of the BERT encoder's F16 and F32 projections over many rows: LDS-tiled, on the 16-bit
// matrix cores (bert.hip launches it; few rows take the direct-load kernel there).
//
// Operands are kept in the order the matrix cores read them ("operand order"): per 32-row tile and
// step of 16 K values PL chunks of 1 KB, in which lane L = 32 g + i holds row i's values
// [8 g, 8 g + 8) of the step. PL = 1: fp16 values (F16 weights and the activations that meet them,
// as ggml-cpu rounds them). PL = 3: fp32 values as three bf16 planes x = h + m + l, exact (each
// takes 8 of the 24 significant bits; bf16 has the range of fp32), so that an F32 product
//   x * w = hh + (hm + mh) + (mm + hl + lh)
// is six v_mfma_f32_32x32x16_bf16 with fp32 accumulation. What is left out, ml + lm + ll, is at
// most 2^-24 of the product (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|), the size of one fp32 rounding of it, and
// 2^-27.5 of it rms (values uniform in [1, 2)). The five small products have accumulators of
// their own, so the large sum is rounded once per 16 K values; the fp32 matrix instruction rounds
// once per 2. The bf16 matrix cores run 16 times as fast as the fp32 ones, six products 2.7 times.
#pragma once
#include "common.h"

namespace gsvk {

typedef _Float16 bv8h __attribute__((ext_vector_type(8)));
typedef __bf16 bv8b __attribute__((ext_vector_type(8)));
typedef float bv16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint16_t bg_lds;

// Offset (in 2-byte values) of element (r, k) of plane 0 of an [R][K] matrix of PL planes in the
// operand order, K % 16 == 0; plane p is 512 p further. Rows are padded to BG_ROW_PAD.
constexpr int BG_ROW_PAD = 128;
template <int PL>
__host__ __device__ inline int64_t bt_off(int64_t r, int64_t k, int64_t K) {
    return (((r >> 5) * (K >> 4) + (k >> 4)) * PL << 9) + (((((k >> 3) & 1) << 5) | (r & 31)) << 3) + (k & 7);
}

// x = h + m + l in bf16 (nearest even each; exact down to the bf16 subnormals). Values that would
// round up to infinity are cut instead; infinities and NaNs go into h alone.
__device__ __forceinline__ void split3(float x, uint16_t & h, uint16_t & m, uint16_t & l) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x), a = u & 0x7fffffffu;
    const uint32_t cut = (u >> 16) | (a > 0x7f800000u ? 0x40u : 0u);
    h = a >= 0x7f7f8000u ? (uint16_t) cut : __builtin_bit_cast(uint16_t, (__bf16) x);
    float r = x - __builtin_bit_cast(float, (uint32_t) h << 16);
    r = a >= 0x7f800000u ? 0.0f : r;
    const __bf16 mb = (__bf16) r;
    m = __builtin_bit_cast(uint16_t, mb);
    l = __builtin_bit_cast(uint16_t, (__bf16) (r - (float) mb));
}

// The same for a pair of values below 2^127 (an infinity gives NaN in m and l).
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t & h, uint32_t & m, uint32_t & l) {
    typedef __bf16 v2b __attribute__((ext_vector_type(2)));
    const auto pk = [](float a, float b) { return __builtin_bit_cast(uint32_t, v2b{(__bf16) a, (__bf16) b}); };
    const auto lo = [](uint32_t u) { return __builtin_bit_cast(float, u << 16); };
    const auto hi = [](uint32_t u) { return __builtin_bit_cast(float, u & 0xffff0000u); };
    h = pk(x0, x1);
    const float r0 = x0 - lo(h), r1 = x1 - hi(h);
    m = pk(r0, r1);
    l = pk(r0 - lo(m), r1 - hi(m));
}

// The e-th of the six products of a (planes of an operand A) and b (of an operand B), the smallest
// first; 5 is the large one.
__device__ __forceinline__ bv16f mfma3(int e, const uint4 (&a)[3], const uint4 (&b)[3], bv16f acc) {
    constexpr int qa[6] = {0, 2, 1, 0, 1, 0}, qb[6] = {2, 0, 1, 1, 0, 0};
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bv8b, a[qa[e]]), __builtin_bit_cast(bv8b, b[qb[e]]), acc, 0, 0, 0);
}

// Store N (4 or 8, aligned) consecutive k values of a row as fp16 / as the three planes.
template <int N>
__device__ __forceinline__ void store_op16(uint16_t * dst, const float * y) {
    uint32_t w[N / 2];
#pragma unroll
    for (int j = 0; j < N / 2; j++) w[j] = (uint32_t) f2h(y[2 * j]) | ((uint32_t) f2h(y[2 * j + 1]) << 16);
    if constexpr (N == 8)
        *reinterpret_cast<uint4 *>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    else
        *reinterpret_cast<uint2 *>(dst) = make_uint2(w[0], w[1]);
}
template <int N>
__device__ __forceinline__ void store_op3(uint16_t * dst, const float * y) {
    uint16_t s[3][N];
#pragma unroll
    for (int j = 0; j < N; j++) split3(y[j], s[0][j], s[1][j], s[2][j]);
#pragma unroll
    for (int p = 0; p < 3; p++) {
        uint32_t w[N / 2];
#pragma unroll
        for (int j = 0; j < N / 2; j++) w[j] = (uint32_t) s[p][2 * j] | ((uint32_t) s[p][2 * j + 1] << 16);
        if constexpr (N == 8)
            *reinterpret_cast<uint4 *>(dst + 512 * p) = make_uint4(w[0], w[1], w[2], w[3]);
        else
            *reinterpret_cast<uint2 *>(dst + 512 * p) = make_uint2(w[0], w[1]);
    }
}

// Output stage of the BERT GEMMs. With a K slice per workgroup (slices > 1) only y is written:
// slice z of the sum to y + z * pstride (partial rows, summed by their consumer).
struct BgOut {
    float * y;            // [M][N] fp32, or null
    int64_t pstride;      // floats between partial slices
    const float * bias;   // added before the activation, or null
    int gelu;             // y = gelu_erf(y + bias) (the add_act of src/gsv_bert.cpp:151-153)
    uint16_t * y16;       // fp16 copy (nearest even) in the operand order (bt_off<1>), or null
    uint16_t * y3;        // three-plane copy in the operand order (bt_off<3>), or null
};

__device__ __forceinline__ float bert_gelu(float y) { return 0.5f * y * (1.0f + erff(y * 0.70710678118654752440f)); }

// A wave's direct load of 1 KB: lane L's 16 bytes at base + off to lds + 16 L. In asm, since the
// compiler waits for every direct load in flight before any LDS read that it cannot tell apart
// from their targets, which would leave one stage in flight instead of NBUF - 1. (No outputs; the
// waits are GSVK_BG_WAIT's, and a wait that the compiler counts without these loads only waits
// longer. The s_nop is the wait state between a write of m0 and a load that reads it.)
__device__ __forceinline__ void bg_load_lds(const uint16_t * base, uint32_t off, uint16_t * lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"((uint32_t) (uintptr_t) (bg_lds *) lds), "v"(off), "s"(base)
                 : "memory");
}

// wait until at most n of this wave's vector-memory operations are outstanding and none of its LDS
// operations (gfx9 encoding: vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8, expcnt not waited on)
#define GSVK_BG_WAIT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | ((((n) >> 4) & 3) << 14) | (0x7 << 4))

// Y[M][N] (or a K slice of it) = X[M][K] . W[N][K]^T. Workgroup: WM x WN waves, each TM x TN MFMA
// tiles of 32 x 32; K streams through LDS in stages of KS steps by direct global -> LDS loads,
// NBUF buffers deep (NBUF - 1 stages in flight), one barrier per stage. Before, 64 x 32 tiles without sharing read 0.9 GB through
// the L2 per FFN1 of 2265 rows; 128 x 128 tiles read 0.3 GB. Measured (fp32 output, us, before -> now):
// fp16 2265 rows N 4096 K 1024 52 -> 32, N 1024 K 4096 49 -> 36; planes 564 rows N 4096 K 1024 79 -> 34,
// N 1024 K 4096 95 -> 33. The matrix cores are busy for 0.22 to 0.31 (fp16) and 0.43 (planes) of the CUs'
// time, the waves wait for a third to half of theirs (counters): the loads and their overlap bound it, not
// the products. A chunk is one load instruction of a wave and one conflict-free 16-byte read per lane
// (SQ_LDS_BANK_CONFLICT 0). The weights are the MFMA's A operand, so a lane holds 4
// consecutive columns of one row per register quad and the epilogue stores from registers.
template <int PL, int TM, int TN, int WM, int WN, int KS, int NBUF>
__global__ void __launch_bounds__(WM * WN * 64) k_bert_gemm_lds(const uint16_t * __restrict__ X,
                                                                const uint16_t * __restrict__ W, int M, int N, int K,
                                                                int slices, int col_major, BgOut o) {
    constexpr int NW = WM * WN, BMT = TM * WM, BNT = TN * WN;   // tiles of 32 rows, of 32 columns
    constexpr int CT = KS * PL;                                 // chunks of a tile and stage, consecutive in memory
    constexpr int CH = CT * (BMT + BNT), CPW = CH / NW;         // chunks of a stage, per wave
    static_assert(CH % NW == 0 && CPW * (NBUF - 1) < 64, "whole chunks per wave, countable by vmcnt");
    __shared__ __align__(16) uint16_t s_ch[NBUF][CH * 512];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    // Workgroup ids go round-robin to the 8 XCDs. Renumbered so that each XCD takes a contiguous
    // run of tiles: with col_major the runs share the XCD's columns (weights), else its rows.
    const int nx = N / (32 * BNT), ny = (M + 32 * BMT - 1) / (32 * BMT), tiles = nx * ny;
    int t;
    {
        const int total = (int) gridDim.x, b = (int) blockIdx.x, per = (total + 7) / 8;
        const int tall = total % 8 == 0 ? 8 : total % 8, xcd = b % 8, loc = b / 8;
        t = xcd < tall ? xcd * per + loc : tall * per + (xcd - tall) * (per - 1) + loc;
    }
    const int p = t / tiles;
    t -= p * tiles;
    const int tx = col_major ? t / ny : t % nx, ty = col_major ? t % ny : t / nx;
    const int nst = K / 16, ns = nst / slices / KS;             // steps of K, stages of this slice
    const int64_t s0 = (int64_t) p * (nst / slices);
    const uint16_t * src[CPW];
#pragma unroll
    for (int j = 0; j < CPW; j++) {
        const int c = wave * CPW + j, tile = c / CT, u = c % CT;
        const int64_t row_tile = tile < BMT ? (int64_t) ty * BMT + tile : (int64_t) tx * BNT + tile - BMT;
        src[j] = (tile < BMT ? X : W) + ((row_tile * nst + s0) * PL + u) * 512;
    }
    auto issue = [&](int stage, int buf, int j0, int j1) {   // chunks [j0, j1) of the wave's
#pragma unroll
        for (int j = j0; j < j1; j++)
            bg_load_lds(src[j] + (int64_t) stage * (CT * 512), lane * 16, &s_ch[buf][(wave * CPW + j) * 512]);
    };
    const int wm = wave / WN, wn = wave % WN;
    constexpr int NA = PL == 3 ? 2 : 1;
    bv16f acc[NA][TM][TN];
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[a][i][j] = bv16f{};
    const int ox = wm * TM * CT * 512 + lane * 8, ow = (BMT + wn * TN) * CT * 512 + lane * 8;
    uint4 a[2][PL][TN], x[2][PL][TM];
    auto read = [&](int buf, int ks) {
#pragma unroll
        for (int q = 0; q < PL; q++) {
#pragma unroll
            for (int j = 0; j < TN; j++)
                a[ks & 1][q][j] = *reinterpret_cast<const uint4 *>(s_ch[buf] + ow + (j * CT + ks * PL + q) * 512);
#pragma unroll
            for (int i = 0; i < TM; i++)
                x[ks & 1][q][i] = *reinterpret_cast<const uint4 *>(s_ch[buf] + ox + (i * CT + ks * PL + q) * 512);
        }
    };
    // (a stage past the end loads the last one again, so that the wait below counts alike)
#pragma unroll
    for (int b = 0; b < NBUF - 1; b++) issue(min(b, ns - 1), b, 0, CPW);
    int buf = 0;
#pragma unroll 1
    for (int st = 0; st < ns; st++) {
        GSVK_BG_WAIT((NBUF - 2) * CPW);             // this wave's part of the stage has landed
        asm volatile("s_barrier" ::: "memory");   // every wave's has, and the last stage is read
        // a step's operands are read before the products of the step before it, and the stage's
        // direct loads are spread over its steps: issued together they would hold up the reads
        read(buf, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks + 1 < KS) read(buf, ks + 1);
            issue(min(st + NBUF - 1, ns - 1), buf == 0 ? NBUF - 1 : buf - 1, ks * CPW / KS, (ks + 1) * CPW / KS);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (PL == 1) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[0][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(bv8h, a[ks & 1][0][j]),
                                                                             __builtin_bit_cast(bv8h, x[ks & 1][0][i]), acc[0][i][j], 0, 0, 0);
            } else {
                constexpr int qa[6] = {0, 2, 1, 0, 1, 0}, qx[6] = {2, 0, 1, 1, 0, 0};   // the smallest first
#pragma unroll
                for (int e = 0; e < 6; e++)
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[e < 5 ? 1 : 0][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                __builtin_bit_cast(bv8b, a[ks & 1][qa[e]][j]), __builtin_bit_cast(bv8b, x[ks & 1][qx[e]][i]),
                                acc[e < 5 ? 1 : 0][i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        buf = buf == NBUF - 1 ? 0 : buf + 1;
    }
    GSVK_BG_WAIT(0);   // the repeated loads land before the LDS is given back
    // lane (li, lg): row m0 + 32 i + li, columns n0 + 32 j + 8 q + 4 lg + [0, 4)
    const int li = lane & 31, lg = lane >> 5;
    const int n0 = (tx * BNT + wn * TN) * 32 + 4 * lg, m0 = (ty * BMT + wm * TM) * 32 + li;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int col = n0 + 32 * j + 8 * q;
            float4 bv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (o.bias) bv = *reinterpret_cast<const float4 *>(o.bias + col);
            const float b[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int row = m0 + 32 * i;
                if (row >= M) continue;
                float y[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    y[v] = acc[0][i][j][4 * q + v];
                    if constexpr (PL == 3) y[v] = y[v] + acc[NA - 1][i][j][4 * q + v];
                    if (o.bias) y[v] = y[v] + b[v];
                    if (o.gelu) y[v] = bert_gelu(y[v]);
                }
                if (o.y)
                    *reinterpret_cast<float4 *>(o.y + (int64_t) p * o.pstride + (int64_t) row * N + col) =
                        make_float4(y[0], y[1], y[2], y[3]);
                if (o.y16) store_op16<4>(o.y16 + bt_off<1>(row, col, N), y);
                if (o.y3) store_op3<4>(o.y3 + bt_off<3>(row, col, N), y);
            }
        }
}

}  // namespace gsvk
