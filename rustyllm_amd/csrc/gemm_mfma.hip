// gemm_mfma.hip — batched K-quant matrix products on the matrix cores, for
// prefill: y[t][r] = row r of W times token t's Q8_K activation, the batch
// matvec of forward_prefill_batch (matvec_kquant3_batch_into,
// src/simd.rs:3461-3578).  Each (row, token) result is bit-identical to the
// single-token GEMV row: the per-block integer sums are exact, and the f32
// combine is the same expression in the same block order (as the reference's
// x4 kernels are bit-identical to its single-token dots, tests
// src/simd.rs:8540-8608).
//
// v_mfma_i32_32x32x32_i8 lane layout (checked on gfx950): A[m = l%32][k =
// 16*(l/32) + j], B[k][n = l%32], C[i] at m = 8*(i/4) + 4*(l/32) + i%4,
// n = l%32.
// Here m = token and n = weight row: a lane owns one weight row, so its
// scales and minimums are per-lane values, and 16 tokens.
//   Q4_K: two x32 MFMAs per 32-element sub-block on the nibbles times the
//         two base-8 digits of the sub-block scale, accumulated over the
//         block, so isum = sum_j sc_j * C_j (C_j = sum q x) exactly; imin =
//         sum_j m_j * bsums_j is one f16 MFMA per block on the sums of 16
//         quants; value = dx * (d*isum - dmin*imin).
//   Q6_K: two x32 MFMAs per 32 elements on the high and low bytes of
//         sc_g (q - 32), accumulated over the block, so isum = sum_g sc_g *
//         C_g exactly; value = (dx*d) * isum.
// Rows past the end read the last row, tokens past the end the last token or
// the batch's padding rows (batch_rows), and neither is stored.
#pragma once
#include "common.hpp"
#include "gemv.hip"
#include "tile_index.hpp"

namespace rh {

typedef int rh_v4i __attribute__((ext_vector_type(4)));
typedef int rh_v16i __attribute__((ext_vector_type(16)));

struct GemmOut {
    const uint8_t *w;
    int64_t row_stride;
    float *y;
    const float *bias;  // [rows] or null
    int32_t rows;
    int32_t ldy;        // y[t * ldy + r]
    int32_t tiles;      // 128-row tiles up to and including this matrix
};
struct GemmArgs {
    GemmOut m[2];       // (m[1] in two-matrix Q4_K launches)
    int32_t K, T;
    int32_t epi;        // EPI_STORE or EPI_ADD
    const int8_t *xq;   // [batch_rows(T)][K] Q8_K quants, token-major
    const float *dx;    // [K/256][ldx] Q8_K scales, token-minor
    const _Float16 *hs; // [K/256][ldx][16] sums of 16 quants
    int32_t ldx;        // >= T, a multiple of 64
};

// One block of the lane's weight row, as the lane's MFMA B operands need it
// (lane half h = lane / 32 takes k = 16h.. of each 32 elements: half a Q4_K
// sub-block, one Q6_K scale group).
template <int FMT>
struct GemmW;
template <>
struct GemmW<F_Q4_K> {
    uint4 hdr, qs[4];
};
template <>
struct GemmW<F_Q6_K> {
    uint4 ql[4], qh[2];  // [64-byte half g][32 bytes kk], [g]: 16 bytes of this lane half
    uint4 sc;
    uint32_t d;
};

__device__ __forceinline__ void gemm_w_load(GemmW<F_Q4_K> &W, const uint8_t *blk, int half) {
    W.hdr = *(const uint4 *)blk;  // 144-byte blocks of 16-aligned rows
#pragma unroll
    for (int q = 0; q < 4; q++) W.qs[q] = *(const uint4 *)(blk + 16 + 32 * q + 16 * half);
}
__device__ __forceinline__ void gemm_w_load(GemmW<F_Q6_K> &W, const uint8_t *blk, int half) {
#pragma unroll
    for (int g = 0; g < 2; g++) {
        W.qh[g] = ld16(blk + 128 + 32 * g + 16 * half);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) W.ql[2 * g + kk] = ld16(blk + 64 * g + 32 * kk + 16 * half);
    }
    W.sc = ld16(blk + 192);
    W.d = ld2(blk + 208);
}

// LDS activation tile: one block (256 quants) of each of the workgroup's
// tokens, rows padded to 272 bytes so the 32 token rows one MFMA operand read
// touches start 4 banks apart.
#define GEMM_XS 272

typedef unsigned short rh_u16x2 __attribute__((ext_vector_type(2)));

// Each byte of the four dwords of x (nibbles, < 16) times s (< 8): one packed
// 16-bit multiply per dword, exact because no byte product (< 128) carries
// into the next byte.
__device__ __forceinline__ rh_v4i bytes_times(const rh_v4i &x, int s) {
    const rh_u16x2 m = {(unsigned short)s, (unsigned short)s};
    rh_v4i r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int xi = x[i];  // a plain int (a bit-cast of the element expression itself reads element 0)
        r[i] = __builtin_bit_cast(int, __builtin_bit_cast(rh_u16x2, xi) * m);
    }
    return r;
}

// Batch products: a workgroup is 128 weight rows (a wave 32) by 32 NT tokens.
//
// Q4_K: the sub-block scale (6 bits) enters the B operand as two digits, sc = 8 (sc
// >> 3) + (sc & 7), each digit times a nibble fitting a signed byte, so the
// MFMAs accumulate the whole block: isum = 8 hi + lo = sum_j sc_j C_j exactly.
// The minimums' sum imin = sum_j m_j (sum of sub-block j) is one 32x32x16 f16
// MFMA on the sums of 16 quants that the quantizers leave: |sum| <= 2048 and
// m <= 63 are exact in f16 and every partial sum is an integer below 2^22, so
// the f32 result is the integer (exactness of such sums checked on the
// device), and it arrives as the float the combine wants.
//
// Per 32 x 32 outputs and block the VALU does the reference's combine, 7
// operations on 16 elements, which nothing can fold, and the wave decodes its
// 32 rows once, about 150 instructions, for its NT token tiles: the digits stay
// in 64 registers.  The activation tile (quants, sums, scales) is double-buffered in
// LDS and shared by the four waves; the next block's comes through registers, a
// few 16-byte pieces per token tile a block ahead (loaded at the tile they are
// stored after, the 28672 x 4096 product took 176 us instead of 160), and its
// weights straight after the digits are made.  One barrier per block.
//
// Bound by the VALU, Q4_K: 200 instructions per 32 x 32 outputs and block with
// NT = 2 (390 with a minimum MFMA per sub-block and one token tile), 62% busy by
// the counters, the matrix cores 37%; the waits are the barrier and the start of
// each tile.  Gate and up of an 8B-class model, 28672 x 4096, 512 tokens in one
// launch: 161 us (747 TOP/s); two launches of the one-tile kernel before, 244.
// Q6_K: the row decode is 330 instructions, a tile 80: with a multiply-add per
// scale group and output instead (430 per tile), 4096 x 14336 and 14336 x 4096,
// 512 tokens took 242 and 213 us, now 164 and 163 (367 TOP/s).  Measured and
// dropped: four token tiles (spills at two waves per SIMD: 189 us); each row
// tile's token tiles on one XCD (160).
typedef _Float16 rh_v8h __attribute__((ext_vector_type(8)));
typedef float rh_v16f __attribute__((ext_vector_type(16)));
typedef float rh_v4f __attribute__((ext_vector_type(4)));

// One block of the lane's Q4_K row as MFMA B operands: per 64 weights the low
// nibbles times the high and low scale digit, then the high nibbles likewise;
// the minimums of this lane half's eight groups of 16 (sub-blocks 4 half .. +
// 3, each twice); d and dmin.
struct Q4kOps {
    rh_v4i dig[4][4];
    rh_v8h bm;
    float d, dmin;
};
__device__ __forceinline__ void q4k_decode(Q4kOps &O, const GemmW<F_Q4_K> &W, int half) {
    const uint4 hdr = W.hdr;
    O.d = h2f((uint16_t)hdr.x);
    O.dmin = h2f((uint16_t)(hdr.x >> 16));
    // scales and minimums of the eight sub-blocks, one per byte
    const uint32_t sc03 = hdr.y & 0x3F3F3F3Fu, sc47 = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
    const uint32_t mn = half ? ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u) : hdr.z & 0x3F3F3F3Fu;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t sw = q < 2 ? sc03 : sc47;
        const int s0 = (sw >> (16 * (q & 1))) & 0xFF, s1 = (sw >> (16 * (q & 1) + 8)) & 0xFF;
        const uint32_t w4[4] = {W.qs[q].x, W.qs[q].y, W.qs[q].z, W.qs[q].w};
        rh_v4i lo, hi;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = (int)(w4[i] & 0x0F0F0F0Fu);
            hi[i] = (int)((w4[i] >> 4) & 0x0F0F0F0Fu);
        }
        O.dig[q][0] = bytes_times(lo, s0 >> 3);
        O.dig[q][1] = bytes_times(lo, s0 & 7);
        O.dig[q][2] = bytes_times(hi, s1 >> 3);
        O.dig[q][3] = bytes_times(hi, s1 & 7);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const _Float16 m = (_Float16)(float)((mn >> (8 * i)) & 0xFF);
        O.bm[2 * i] = m;
        O.bm[2 * i + 1] = m;
    }
}

// The block's values dx (d isum - dmin imin) of 32 rows x 32 tokens: xr the
// lane's token row of the LDS tile (+ 16 half), hs its sums, dv(g) the scales
// of tokens 8 g + 4 half ..; out(i, value) takes C element i's.
template <class Dv, class Out>
__device__ __forceinline__ void q4k_tile(const Q4kOps &O, const int8_t *xr, rh_v8h hs, Dv dv, Out out) {
    rh_v16i hi = {}, lo = {};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const rh_v4i a0 = *(const rh_v4i *)(xr + 64 * q), a1 = *(const rh_v4i *)(xr + 64 * q + 32);
        hi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0, O.dig[q][0], hi, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0, O.dig[q][1], lo, 0, 0, 0);
        hi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, O.dig[q][2], hi, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, O.dig[q][3], lo, 0, 0, 0);
    }
    const rh_v16f im = __builtin_amdgcn_mfma_f32_32x32x16_f16(hs, O.bm, rh_v16f{}, 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const rh_v4f dx = dv(g);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 4 * g + r;
            const float t1 = O.d * (float)((hi[i] << 3) + lo[i]);
            const float t2 = O.dmin * im[i];
            out(i, dx[r] * (t1 - t2));
        }
    }
}

// One block of the lane's Q6_K row as MFMA B operands.  Lane half h holds
// elements 16 h .. + 15 of every 32, i.e. one scale group, so the products
// sc (q - 32) (at most 4096 in magnitude) can be the operand: as the signed
// bytes hi and lo of 256 hi + lo, one pair per 32 elements.
struct Q6kOps {
    rh_v4i hi[8], lo[8];
    float d;
};
__device__ __forceinline__ void q6k_decode(Q6kOps &O, const GemmW<F_Q6_K> &W, int half) {
    O.d = h2f((uint16_t)W.d);
    const uint32_t sc4[4] = {W.sc.x, W.sc.y, W.sc.z, W.sc.w};
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const uint32_t qh4[4] = {W.qh[g].x, W.qh[g].y, W.qh[g].z, W.qh[g].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint4 ql = W.ql[2 * g + (k & 1)];
            const uint32_t ql4[4] = {ql.x, ql.y, ql.z, ql.w};
            // scale 8 g + 2 k + half; p + 128 = sc q + (128 - 32 sc), 16 bits each
            const int sc = (int)(int8_t)(sc4[2 * g + (k >> 1)] >> (16 * (k & 1) + 8 * half));
            const unsigned short su = (unsigned short)sc, cu = (unsigned short)(128 - 32 * sc);
            const rh_u16x2 s2 = {su, su}, c2 = {cu, cu};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t hb = (k < 2 ? qh4[i] << (4 - 2 * k) : qh4[i] >> (2 * k - 4)) & 0x30303030u;
                const uint32_t q = ((k < 2 ? ql4[i] : ql4[i] >> 4) & 0x0F0F0F0Fu) | hb;
                const uint32_t qe = q & 0x00FF00FFu;
                const rh_u16x2 qo = __builtin_bit_cast(rh_u16x2, q) >> 8;
                const uint32_t pe = __builtin_bit_cast(uint32_t, __builtin_bit_cast(rh_u16x2, qe) * s2 + c2);
                const uint32_t po = __builtin_bit_cast(uint32_t, qo * s2 + c2);
                // bytes of (po:pe): 0..3 are pe's, 4..7 po's
                O.hi[4 * g + k][i] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
                O.lo[4 * g + k][i] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
            }
        }
    }
}

// The block's values (dx d) isum of 32 rows x 32 tokens: xr the lane's token
// row of the LDS tile (+ 16 half); dv and out as q4k_tile's.
template <class Dv, class Out>
__device__ __forceinline__ void q6k_tile(const Q6kOps &O, const int8_t *xr, Dv dv, Out out) {
    rh_v16i hi = {}, lo = {};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const rh_v4i a = *(const rh_v4i *)(xr + 32 * e);
        hi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, O.hi[e], hi, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, O.lo[e], lo, 0, 0, 0);
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const rh_v4f dx = dv(g);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 4 * g + r;
            out(i, (dx[r] * O.d) * (float)((hi[i] << 8) + lo[i]));
        }
    }
}

template <int FMT>
struct GemmOps {
    typedef Q6kOps type;
};
template <>
struct GemmOps<F_Q4_K> {
    typedef Q4kOps type;
};

constexpr int gemm_kq_buf(int nt) { return 32 * nt * (GEMM_XS + 32 + 4); }
constexpr int gemm_kq_lds(int nt) { return 2 * gemm_kq_buf(nt); }

template <int FMT, int NT>
__global__ __launch_bounds__(256, 2) void gemm_kq_mfma_kernel(GemmArgs A) {
    extern __shared__ __align__(16) int8_t s_xt[];  // [2]: quants [TOK][GEMM_XS], sums [TOK][16] f16, scales [TOK]
    constexpr int TOK = 32 * NT, HS0 = TOK * GEMM_XS, DX0 = HS0 + TOK * 32, BUF = gemm_kq_buf(NT);
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x, by = blockIdx.y;
    const bool m1 = bx >= A.m[0].tiles;
    const int rows = m1 ? A.m[1].rows : A.m[0].rows;
    const int r0 = (bx - (m1 ? A.m[0].tiles : 0)) * 128 + 32 * wave;
    const int t0 = by * TOK;
    const uint8_t *wr = (m1 ? A.m[1].w : A.m[0].w) +
                        (int64_t)min(r0 + n, rows - 1) * (m1 ? A.m[1].row_stride : A.m[0].row_stride);
    const int nb = A.K >> 8;
    // activation pieces (gemm_x_lane); tokens past the batch read the rows that
    // batch_rows adds for them (their outputs are not stored)
    const __amdgpu_buffer_rsrc_t xres =
        __builtin_amdgcn_make_buffer_rsrc((void *)(A.xq + (int64_t)t0 * A.K), (short)0, TOK * A.K, 0x00020000);
    const int xoff = gemm_x_lane(tid, A.K), xdst = (tid >> 4) * GEMM_XS + 16 * (tid & 15);
    const int ht = min(t0 + min(tid, 2 * TOK - 1) / 2, A.T - 1), dt = min(t0 + min(tid, TOK - 1), A.T - 1);
    auto load_x = [&](int b, int j) {
        return __builtin_amdgcn_raw_buffer_load_b128(xres, xoff, gemm_x_step(j, b, A.K), 0);
    };
    typedef decltype(__builtin_amdgcn_raw_buffer_load_b128(xres, 0, 0, 0)) piece_t;
    constexpr int BB = FMT == F_Q4_K ? 144 : 210;
    GemmW<FMT> W;
    auto load_w = [&](int b) { gemm_w_load(W, wr + (int64_t)b * BB, half); };
    rh_v4i hsr;
    float dxr = 0.0f;
    auto load_hd = [&](int b) {
        if (FMT == F_Q4_K && tid < 2 * TOK) hsr = *(const rh_v4i *)(A.hs + ((int64_t)b * A.ldx + ht) * 16 + 8 * (tid & 1));
        if (tid < TOK) dxr = A.dx[(int64_t)b * A.ldx + dt];
    };
    auto store_hd = [&](int8_t *buf) {
        if (FMT == F_Q4_K && tid < 2 * TOK) *(rh_v4i *)(buf + HS0 + 16 * tid) = hsr;
        if (tid < TOK) *(float *)(buf + DX0 + 4 * tid) = dxr;
    };
    piece_t st[2 * NT];
    load_w(0);
    load_hd(0);
#pragma unroll
    for (int j = 0; j < 2 * NT; j++) st[j] = load_x(0, j);
#pragma unroll
    for (int j = 0; j < 2 * NT; j++) *(piece_t *)(s_xt + xdst + 16 * j * GEMM_XS) = st[j];
    store_hd(s_xt);
    load_hd(min(1, nb - 1));
#pragma unroll
    for (int j = 0; j < 2 * NT; j++) st[j] = load_x(min(1, nb - 1), j);
    float acc[NT][16];
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[tt][i] = 0.0f;
    __syncthreads();
    for (int b = 0; b < nb; b++) {
        const int8_t *cur = s_xt + (b & 1) * BUF;
        int8_t *nxt = s_xt + ((b + 1) & 1) * BUF;
        const int bn = min(b + 1, nb - 1);  // (the last block stages itself again, unread)
        typename GemmOps<FMT>::type O;
        if constexpr (FMT == F_Q4_K)
            q4k_decode(O, W, half);
        else
            q6k_decode(O, W, half);
        load_w(bn);
        // the next block's activations, loaded a block ago, then the one after
        store_hd(nxt);
#pragma unroll
        for (int j = 0; j < 2 * NT; j++) *(piece_t *)(nxt + xdst + 16 * j * GEMM_XS) = st[j];
        const int b2 = min(b + 2, nb - 1);
        load_hd(b2);
#pragma unroll
        for (int j = 0; j < 2 * NT; j++) st[j] = load_x(b2, j);
#pragma unroll
        for (int tt = 0; tt < NT; tt++) {
            // the reference's per-block combine, accumulated in block order
            const int8_t *xr = cur + (32 * tt + n) * GEMM_XS;
            const auto dv = [&](int g) { return *(const rh_v4f *)(cur + DX0 + 4 * (32 * tt + 8 * g + 4 * half)); };
            const auto out = [&](int i, float v) { acc[tt][i] += v; };
            if constexpr (FMT == F_Q4_K)
                q4k_tile(O, xr + 16 * half, *(const rh_v8h *)(cur + HS0 + (32 * tt + n) * 32 + 16 * half), dv, out);
            else
                q6k_tile(O, xr + 16 * half, dv, out);
        }
        __syncthreads();
    }
    if (r0 + n >= rows) return;
    const float *bp = m1 ? A.m[1].bias : A.m[0].bias;
    const float bias = bp ? bp[r0 + n] : 0.0f;
    const int ldy = m1 ? A.m[1].ldy : A.m[0].ldy;
    float *y = (m1 ? A.m[1].y : A.m[0].y) + r0 + n;
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = t0 + 32 * tt + 8 * (i >> 2) + 4 * half + (i & 3);
            if (t >= A.T) continue;
            float v = acc[tt][i];
            if (bp) v = v + bias;
            if (A.epi == EPI_ADD)
                y[(int64_t)t * ldy] += v;
            else
                y[(int64_t)t * ldy] = v;
        }
}

// The same products with the blocks of K split over the workgroup's four
// waves, for launches with too few (row tile, token tile) pairs to fill the
// chip: one workgroup per 32 weight rows x 32 tokens, wave w
// computing blocks w, w+4, w+8, ...  Each wave stages its own block's
// activations in its own LDS tile, computes the block's per-output value
// exactly as the unsplit kernel does, and leaves the 16 values of each lane in
// LDS; after a barrier, wave w adds the round's values of C elements 4w..4w+3
// to its accumulators in block order (a barrier before the next round's values
// are written keeps them until every wave has read these).  Every output is
// therefore the same sum of the same per-block values in the same order.
template <int FMT>
__global__ __launch_bounds__(256) void gemm_kq_mfma_ks_kernel(GemmArgs A) {
    __shared__ __align__(16) int8_t s_xs[4][32 * GEMM_XS];  // per wave: 32 token rows of one block
    __shared__ float s_v[4][16][64];                        // [wave][C element][lane]
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = blockIdx.x * 32, t0 = blockIdx.y * 32;
    const int row = min(r0 + n, A.m[0].rows - 1);
    const uint8_t *wr = A.m[0].w + (int64_t)row * A.m[0].row_stride;
    const int nb = A.K >> 8, rounds = (nb + 3) >> 2;
    constexpr int BB = FMT == F_Q4_K ? 144 : 210;
    // activation pieces of the wave's block: lane -> (token, 16-byte part),
    // 16 lanes per token row, 4 rows per load
    const int8_t *xsrc[8];
    int xdst[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int p = lane + 64 * j, tok = p >> 4, part = p & 15;
        xsrc[j] = A.xq + (int64_t)min(t0 + tok, A.T - 1) * A.K + 16 * part;
        xdst[j] = tok * GEMM_XS + 16 * part;
    }
    int8_t *xs = s_xs[wave];
    int b = min(wave, nb - 1);
    // a block's scales and sums (rows up to ldx, a multiple of 64, exist)
    rh_v4f dv[4];
    rh_v8h hs;
    auto load_hd = [&](int bl) {
#pragma unroll
        for (int g = 0; g < 4; g++) dv[g] = *(const rh_v4f *)(A.dx + (int64_t)bl * A.ldx + t0 + 4 * half + 8 * g);
        if constexpr (FMT == F_Q4_K) hs = *(const rh_v8h *)(A.hs + ((int64_t)bl * A.ldx + t0 + n) * 16 + 8 * half);
    };
    GemmW<FMT> W;
    gemm_w_load(W, wr + (int64_t)b * BB, half);
    load_hd(b);
    {
        uint4 st[8];
#pragma unroll
        for (int j = 0; j < 8; j++) st[j] = *(const uint4 *)(xsrc[j] + 256 * b);
#pragma unroll
        for (int j = 0; j < 8; j++) *(uint4 *)(xs + xdst[j]) = st[j];
    }
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int it = 0;
    do {  // (rounds >= 1; a loop that might not run would draw the first loads to after the staging's waits)
        b = 4 * it + wave;
        const bool have = b < nb;
        const int bn = min(b + 4, nb - 1);  // the wave's next block (clamped; unused past the end)
        GemmW<FMT> Wn;
        gemm_w_load(Wn, wr + (int64_t)bn * BB, half);
        float v[16] = {};
        if (have) {
            if constexpr (FMT == F_Q4_K) {
                Q4kOps O;
                q4k_decode(O, W, half);
                q4k_tile(O, xs + n * GEMM_XS + 16 * half, hs, [&](int g) { return dv[g]; },
                         [&](int i, float val) { v[i] = val; });
            } else {
                Q6kOps O;
                q6k_decode(O, W, half);
                q6k_tile(O, xs + n * GEMM_XS + 16 * half, [&](int g) { return dv[g]; },
                         [&](int i, float val) { v[i] = val; });
            }
        }
        // the next block's scales, sums and activations, in flight over the barrier
        // (issued after this block's products, so that they hold no registers
        // there; with the scales and sums loaded at the top of their own round the
        // products waited for them and the next weights: 1024 x 14336, 8 tokens 27.9
        // us, now 24.3)
        load_hd(bn);
        rh_v4i st[8];
#pragma unroll
        for (int j = 0; j < 8; j++) st[j] = *(const rh_v4i *)(xsrc[j] + 256 * bn);
        __syncthreads();  // every wave has read the previous round's values
        if (have) {
#pragma unroll
            for (int i = 0; i < 16; i++) s_v[wave][i][lane] = v[i];
        }
        // (this wave's own tile: its LDS reads above complete before these
        // writes, in program order)
#pragma unroll
        for (int j = 0; j < 8; j++) *(rh_v4i *)(xs + xdst[j]) = st[j];
        __syncthreads();
        // the round's blocks in order, for this wave's four C elements
#pragma unroll
        for (int w2 = 0; w2 < 4; w2++) {
            if (4 * it + w2 >= nb) break;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += s_v[w2][4 * wave + e][lane];
        }
        W = Wn;
    } while (++it < rounds);
    if (r0 + n >= A.m[0].rows) return;
    const float bias = A.m[0].bias ? A.m[0].bias[r0 + n] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int i = 4 * wave + e;
        const int t = t0 + 8 * (i >> 2) + 4 * half + (i & 3);
        if (t >= A.T) continue;
        float *yp = A.m[0].y + (int64_t)t * A.m[0].ldy + r0 + n;
        float v = acc[e];
        if (A.m[0].bias) v = v + bias;
        if (A.epi == EPI_ADD)
            *yp += v;
        else
            *yp = v;
    }
}

}  // namespace rh
