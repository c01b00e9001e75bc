// prefill_moe.hip — batched prefill for the gpt-oss resident decoder.  The
// reference prefills gpt-oss token by token (forward_prefill_gpt_oss,
// src/model.rs:10286, i.e. forward_hidden_gpt_oss_impl without the final
// norm); here a chunk of T prompt tokens goes through each layer together, so
// each dense matrix is read once per token group and each expert matrix once
// per group of the tokens routed to it, while every token's arithmetic is its
// decode step's: the same dot orders, RMSNorm, RoPE, attention, SwiGLU and
// slot-ordered combine.  The kernels here add a token dimension to the decode
// step's kernels; the host side (r_prefill_chunk_moe) strings them together.
#pragma once
#include "attention_exact.hip"
#include "common.hpp"
#include "gemv.hip"
#include "moe.hip"
#include "ops.hip"

namespace rh {

// rms_norm_into of T rows, f32 out: rmsnorm_q8k_kernel's arithmetic per row.
// grid (ceil(n/256), T), dynamic LDS n floats; n % 4 == 0.
__global__ __launch_bounds__(256) void rmsnorm_f32_batch_kernel(const float *x, const float *w, float eps, int n,
                                                                float *xn) {
    const int64_t t = blockIdx.y;
    rmsnorm_row(x + t * n, w, eps, n, xn + t * n, XQ{});
}

// Q8_0 rows for T tokens; each (row, token) is exactly the single-token
// kernel's value: F32, dot_q8_0_f32_avx2 as gemv_q8_0_f32x_kernel (eight
// lane accumulators acc_j = fma(d*q, x[32b + 8i + j], acc_j)); otherwise
// dot_q8_0_q8k_avx2 as gemv_q8_0_pipe_kernel (acc_j = fma(dx*d, s_j, acc_j),
// s_j the exact dot of bytes 4j..4j+3); then hsum_avx, bias, store or add.
// A workgroup is 32 rows (4 waves x 8 rows x 8 lanes, lane j accumulator j)
// by TG tokens whose activations are staged in LDS: F32 float [TG][K]; Q8_K
// int8 [TG][K] then the scales float [TG][K/256].  grid (ceil(rows/32),
// ceil(T/TG)).
struct Q80BatchArgs {
    const uint8_t *w;
    int64_t row_stride;
    int32_t rows, K, T, epi;
    const float *x;    // F32: [T][K]
    const int8_t *qs;  // Q8_K: quants [T][K], scales [K/256][ldx] (token-minor)
    const float *dx;
    int32_t ldx;
    const float *bias;
    float *y;  // [T][ldy]
    int32_t ldy;
};

template <bool F32, int TG>
__global__ __launch_bounds__(256) void gemv_q8_0_batch_kernel(Q80BatchArgs A) {
    extern __shared__ __align__(16) uint8_t s_act[];
    const int K = A.K, nb = K >> 5, tid = threadIdx.x;
    const int t0 = blockIdx.y * TG, tn = min(TG, A.T - t0);
    if (F32) {
        float4 *sx = (float4 *)s_act;
        const int k4 = K / 4;
        for (int i = tid; i < TG * k4; i += 256) {
            const int z = i / k4, c = i - z * k4;
            sx[i] = z < tn ? ((const float4 *)(A.x + (int64_t)(t0 + z) * K))[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    } else {
        int4 *sq = (int4 *)s_act;
        float *sd = (float *)(s_act + (size_t)TG * K);
        const int k16 = K / 16, nsb = K / 256;
        for (int i = tid; i < TG * k16; i += 256) {
            const int z = i / k16, c = i - z * k16;
            sq[i] = z < tn ? ((const int4 *)(A.qs + (int64_t)(t0 + z) * K))[c] : make_int4(0, 0, 0, 0);
        }
        for (int i = tid; i < TG * nsb; i += 256) {
            const int z = i / nsb, b = i - z * nsb;
            sd[i] = z < tn ? A.dx[(int64_t)b * A.ldx + t0 + z] : 0.0f;
        }
    }
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6, j = lane & 7;
    const int row = blockIdx.x * 32 + wave * 8 + (lane >> 3);
    const bool ok = row < A.rows;
    const uint8_t *rp = A.w + (int64_t)(ok ? row : 0) * A.row_stride;
    float acc[TG];
#pragma unroll
    for (int z = 0; z < TG; z++) acc[z] = 0.0f;
    for (int b = 0; b < nb; b++) {
        const uint8_t *blk = rp + b * 34;
        const float d = ldh(blk);
        const uint4 q0 = ld16(blk + 2), q1 = ld16(blk + 18);
        if (F32) {
            // byte 8i + j of the 32 quants: dword 2i + j/4, bits 8*(j%4)
            const uint32_t sh = 8u * (uint32_t)(j & 3);
            const bool hi = j >= 4;
            const uint32_t dw[4] = {hi ? q0.y : q0.x, hi ? q0.w : q0.z, hi ? q1.y : q1.x, hi ? q1.w : q1.z};
            float dq[4];
#pragma unroll
            for (int i = 0; i < 4; i++) dq[i] = d * (float)(int)__builtin_amdgcn_sbfe((int)dw[i], sh, 8u);
            const float *sx = (const float *)s_act + b * 32 + j;
#pragma unroll
            for (int z = 0; z < TG; z++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[z] = fmaf(dq[i], sx[(size_t)z * K + 8 * i], acc[z]);
        } else {
            const uint32_t wsel[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
            uint32_t wj = wsel[0];
#pragma unroll
            for (int i = 1; i < 8; i++) wj = j == i ? wsel[i] : wj;
            const int32_t *sq = (const int32_t *)s_act;
            const float *sd = (const float *)(s_act + (size_t)TG * K);
#pragma unroll
            for (int z = 0; z < TG; z++) {
                const float sc = sd[z * (K / 256) + (b >> 3)] * d;
                const int s = sdot4(wj, sq[(size_t)z * (K / 4) + b * 8 + j], 0);
                acc[z] = fmaf(sc, (float)s, acc[z]);
            }
        }
    }
#pragma unroll
    for (int z = 0; z < TG; z++) {
        // hsum_avx: t_i = a_i + a_{i+4}; ((t0+t1) + (t2+t3))
        const float t = acc[z] + __shfl_xor(acc[z], 4, 64);
        const float u = t + __shfl_xor(t, 1, 64);
        float v = u + __shfl_xor(u, 2, 64);
        if (z < tn && ok && j == 0) {
            if (A.bias) v += A.bias[row];
            float *y = A.y + (int64_t)(t0 + z) * A.ldy + row;
            if (A.epi == EPI_ADD)
                *y += v;
            else
                *y = v;
        }
    }
}

// ---- Q8_0 products of a token batch on the matrix cores ----------------------
// y[t][r] for up to three matrices that share their activations (the q/k/v
// projections in one launch: k and v alone would leave half of the CUs idle);
// each (row, token) is exactly the single-token kernel's value.  A workgroup
// is 64 rows by 64 tokens, wave (wr, wt) of it 32 rows by 32 tokens with eight
// accumulators per output, one per AVX2 lane j.  Both operands of a chunk of
// two 32-element blocks are staged in LDS in the form the MFMAs take them
// (double-buffered, loaded through registers a chunk ahead; one barrier per
// chunk), so a weight is decoded once per 64 tokens.
struct Q80GemmArgs {
    Q80BatchArgs m[3];  // epi, x / qs / dx / ldx, K and T are the same in all
    int32_t tiles[3];   // 64-row tiles up to and including matrix i
};
#define Q8G_P 68  // row pitch in LDS, floats: 16-byte reads of 8 rows start on distinct banks

__device__ __forceinline__ Q80BatchArgs q80_gemm_pick(const Q80GemmArgs &G, int &row0) {
    const int bx = blockIdx.x;
    const int i = bx < G.tiles[0] ? 0 : bx < G.tiles[1] ? 1 : 2;
    row0 = 64 * (bx - (i == 0 ? 0 : i == 1 ? G.tiles[0] : G.tiles[1]));
    // member by member: a copy of a run-time element would go through scratch
    Q80BatchArgs A = G.m[0];
    A.w = i == 0 ? A.w : i == 1 ? G.m[1].w : G.m[2].w;
    A.row_stride = i == 0 ? A.row_stride : i == 1 ? G.m[1].row_stride : G.m[2].row_stride;
    A.rows = i == 0 ? A.rows : i == 1 ? G.m[1].rows : G.m[2].rows;
    A.bias = i == 0 ? A.bias : i == 1 ? G.m[1].bias : G.m[2].bias;
    A.y = i == 0 ? A.y : i == 1 ? G.m[1].y : G.m[2].y;
    A.ldy = i == 0 ? A.ldy : i == 1 ? G.m[1].ldy : G.m[2].ldy;
    return A;
}

typedef float q8_v4f __attribute__((ext_vector_type(4)));
typedef float q8_v16f __attribute__((ext_vector_type(16)));

// hsum_avx of the eight accumulators, bias, store or add.  C element i of lane
// (n, h) is (token 8 (i / 4) + 4 h + i % 4, row n).
__device__ __forceinline__ void q80_gemm_store(const Q80BatchArgs &A, const q8_v16f (&acc)[8], int row, int t0, int h) {
    if (row >= A.rows) return;
    const float bias = A.bias ? A.bias[row] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int t = t0 + 8 * (i >> 2) + 4 * h + (i & 3);
        if (t >= A.T) continue;
        float v = ((acc[0][i] + acc[4][i]) + (acc[1][i] + acc[5][i])) + ((acc[2][i] + acc[6][i]) + (acc[3][i] + acc[7][i]));
        if (A.bias) v += bias;
        float *y = A.y + (int64_t)t * A.ldy + row;
        if (A.epi == EPI_ADD)
            *y += v;
        else
            *y = v;
    }
}

// f32 activations (K % 256 != 0): acc_j = fma(d q, x, acc_j) over the elements
// e = j (mod 8) in order.  v_mfma_f32_32x32x2_f32 is two such steps in k order
// (gemm_mxfp4_experts_kernel), so chain j takes elements 16 u + j and 16 u + 8
// + j in MFMA u: lane half h holds elements 8 h .. 8 h + 7 of every 16.  d q is
// exact in f32.  Bound by the matrix cores, 64 clocks per 32 x 32 x 2 products
// (157 TFLOP/s).  Measured: the q, k and v products of gpt-oss-20b (5120 x
// 2880, 1001 tokens) 300 us (98 TFLOP/s), 2253 with gemv_q8_0_batch_kernel.
__global__ __launch_bounds__(256, 2) void gemm_q8_0_f32_kernel(Q80GemmArgs G) {
    __shared__ __align__(16) float s_x[2][64 * Q8G_P], s_w[2][64 * Q8G_P];
    int row0;
    const Q80BatchArgs A = q80_gemm_pick(G, row0);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5, wr = wave & 1, wt = wave >> 1, t0 = blockIdx.y * 64;
    const int K = A.K, nb = K >> 5, nc = (nb + 1) / 2;
    // thread t stages float4 t % 16 of the chunk for tokens t / 16 + 16 j, and
    // quants 8 (t % 4) .. + 7 of row t / 4 of both blocks
    const int c4 = tid & 15, part = tid & 3;
    const float *xr[4];
#pragma unroll
    for (int j = 0; j < 4; j++) xr[j] = A.x + (int64_t)min(t0 + (tid >> 4) + 16 * j, A.T - 1) * K + 4 * c4;
    const uint8_t *wr0 = A.w + (int64_t)min(row0 + (tid >> 2), A.rows - 1) * A.row_stride;
    q8_v4f xs[4];
    uint2 wq[2];
    uint16_t wd[2];
    auto load = [&](int c) {
        const bool in = 64 * c + 4 * c4 < K;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            xs[j] = q8_v4f{0.f, 0.f, 0.f, 0.f};
            if (in) xs[j] = *(const q8_v4f *)(xr[j] + 64 * c);
        }
#pragma unroll
        for (int o = 0; o < 2; o++) {
            const uint8_t *blk = wr0 + (int64_t)min(2 * c + o, nb - 1) * 34;
            wd[o] = ld2(blk);
            wq[o] = ld8(blk + 2 + 8 * part);
        }
    };
    auto store = [&](int c) {
        float *dx = s_x[c & 1] + (tid >> 4) * Q8G_P + 4 * c4;
#pragma unroll
        for (int j = 0; j < 4; j++) *(q8_v4f *)(dx + 16 * j * Q8G_P) = xs[j];
        float *dw = s_w[c & 1] + (tid >> 2) * Q8G_P + 8 * part;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            const float d = h2f(wd[o]);
            q8_v4f a, b;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                a[i] = d * (float)(int8_t)(wq[o].x >> (8 * i));
                b[i] = d * (float)(int8_t)(wq[o].y >> (8 * i));
            }
            *(q8_v4f *)(dw + 32 * o) = a;
            *(q8_v4f *)(dw + 32 * o + 4) = b;
        }
    };
    q8_v16f acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = q8_v16f{};
    load(0);
    store(0);
    load(min(1, nc - 1));
    for (int c = 0; c < nc; c++) {
        __syncthreads();  // chunk c is in LDS; chunk c - 1's reads are done
        if (c + 1 < nc) store(c + 1);
        if (c + 2 < nc) load(c + 2);
        const float *xa = s_x[c & 1] + (32 * wt + n) * Q8G_P + 8 * h;
        const float *wa = s_w[c & 1] + (32 * wr + n) * Q8G_P + 8 * h;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            if (2 * c + o >= nb) break;  // uniform
#pragma unroll
            for (int u = 0; u < 2; u++) {
                q8_v4f a[2], b[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    a[q] = *(const q8_v4f *)(xa + 32 * o + 16 * u + 4 * q);
                    b[q] = *(const q8_v4f *)(wa + 32 * o + 16 * u + 4 * q);
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j >> 2][j & 3], b[j >> 2][j & 3], acc[j], 0, 0, 0);
            }
        }
    }
    q80_gemm_store(A, acc, row0 + 32 * wr + n, t0 + 32 * wt, h);
}

// Q8_K activations (K % 256 == 0): acc_j = fma(dx d, s_j, acc_j) per 32-element
// block, s_j the exact dot of bytes 4 j .. 4 j + 3.  v_mfma_f32_32x32x4_2b_f16
// gives two of the eight s_j at once, as f32 with no conversion: quants are
// exact in f16 and |s_j| <= 2^16; lane half h holds chain j = 2 u + h of MFMA
// u.  Bound by the VALU's 144 multiplies and fused adds per 32 x 32 outputs
// and block (the matrix cores' 4 x 64 clocks run beside them).  Measured: wo
// of gpt-oss-20b (2880 x 4096, 1001 tokens) 212 us, 975 with
// gemv_q8_0_batch_kernel.
typedef _Float16 q8_v4h __attribute__((ext_vector_type(4)));
typedef _Float16 q8_v2h __attribute__((ext_vector_type(2)));
typedef float q8_v32f __attribute__((ext_vector_type(32)));
#define Q8G_HP 72  // row pitch of the f16 operands in LDS, halves (144 bytes)

// four signed bytes as f16: 1024 + (q + 128) by its bit pattern, minus 1152
__device__ __forceinline__ q8_v4h i8x4_to_f16(uint32_t q) {
    const uint32_t u = q ^ 0x80808080u;
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const q8_v2h off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const q8_v2h a = __builtin_bit_cast(q8_v2h, lo) - off, b = __builtin_bit_cast(q8_v2h, hi) - off;
    return q8_v4h{a[0], a[1], b[0], b[1]};
}

__global__ __launch_bounds__(256, 2) void gemm_q8_0_q8k_kernel(Q80GemmArgs G) {
    __shared__ __align__(16) _Float16 s_x[2][64 * Q8G_HP], s_w[2][64 * Q8G_HP];
    __shared__ float s_d[2][2][64];
    int row0;
    const Q80BatchArgs A = q80_gemm_pick(G, row0);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5, wr = wave & 1, wt = wave >> 1, t0 = blockIdx.y * 64;
    const int K = A.K, nc = K >> 6;
    // thread t stages quants 8 (t % 4) .. + 7 of both blocks of token / row t / 4:
    // the first four are chain 2 (t % 4), the others the next
    const int part = tid & 3, r = tid >> 2;
    const int8_t *xr = A.qs + (int64_t)min(t0 + r, A.T - 1) * K + 8 * part;
    const uint8_t *wr0 = A.w + (int64_t)min(row0 + r, A.rows - 1) * A.row_stride;
    uint2 xq[2], wq[2];
    uint16_t wd[2];
    auto load = [&](int c) {
#pragma unroll
        for (int o = 0; o < 2; o++) {
            xq[o] = *(const uint2 *)(xr + 64 * c + 32 * o);
            const uint8_t *blk = wr0 + (int64_t)(2 * c + o) * 34;
            wd[o] = ld2(blk);
            wq[o] = ld8(blk + 2 + 8 * part);
        }
    };
    // LDS row: [block][h][u][4 halves]
    auto store = [&](int c) {
        _Float16 *dx = s_x[c & 1] + r * Q8G_HP + 4 * part, *dw = s_w[c & 1] + r * Q8G_HP + 4 * part;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            *(q8_v4h *)(dx + 32 * o) = i8x4_to_f16(xq[o].x);
            *(q8_v4h *)(dx + 32 * o + 16) = i8x4_to_f16(xq[o].y);
            *(q8_v4h *)(dw + 32 * o) = i8x4_to_f16(wq[o].x);
            *(q8_v4h *)(dw + 32 * o + 16) = i8x4_to_f16(wq[o].y);
            if (part == 0) s_d[c & 1][o][r] = h2f(wd[o]);
        }
    };
    q8_v16f acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = q8_v16f{};
    q8_v4f dt[4];  // the scales of the lane's 16 tokens for the 256-element block in hand
    load(0);
    store(0);
    load(min(1, nc - 1));
    for (int c = 0; c < nc; c++) {
        __syncthreads();  // chunk c is in LDS; chunk c - 1's reads are done
        if ((c & 3) == 0) {
            // ldx is a multiple of 64 >= T: the tile's 64 scales exist
            const float *p = A.dx + (int64_t)(c >> 2) * A.ldx + t0 + 32 * wt + 4 * h;
#pragma unroll
            for (int q = 0; q < 4; q++) dt[q] = *(const q8_v4f *)(p + 8 * q);
        }
        if (c + 1 < nc) store(c + 1);
        if (c + 2 < nc) load(c + 2);
        const _Float16 *xa = s_x[c & 1] + (32 * wt + n) * Q8G_HP + 16 * h;
        const _Float16 *wa = s_w[c & 1] + (32 * wr + n) * Q8G_HP + 16 * h;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            const float d = s_d[c & 1][o][32 * wr + n];
            float sc[16];
#pragma unroll
            for (int i = 0; i < 16; i++) sc[i] = dt[i >> 2][i & 3] * d;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const q8_v4h a = *(const q8_v4h *)(xa + 32 * o + 4 * u), b = *(const q8_v4h *)(wa + 32 * o + 4 * u);
                const q8_v32f s = __builtin_amdgcn_mfma_f32_32x32x4f16(a, b, q8_v32f{}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    acc[2 * u][i] = fmaf(sc[i], s[i], acc[2 * u][i]);
                    acc[2 * u + 1][i] = fmaf(sc[i], s[16 + i], acc[2 * u + 1][i]);
                }
            }
        }
    }
    q80_gemm_store(A, acc, row0 + 32 * wr + n, t0 + 32 * wt, h);
}

// Router selection of T tokens (moe_topk_kernel per token): logits [T][ldl],
// sel / prob [T][k].  grid T.
__global__ __launch_bounds__(64) void moe_topk_batch_kernel(const float *logits, int ldl, int n, int k, int32_t *sel,
                                                            float *prob) {
    const int64_t t = blockIdx.x;
    moe_topk_row(logits + t * ldl, n, k, sel + t * k, prob + t * k);
}

// x[t] += sum over slots r in order of (proj[t k + r] + db[e_r]) * p_r, per
// token (moe_combine_kernel).  grid (ceil(dim/256), T).
__global__ __launch_bounds__(256) void moe_combine_batch_kernel(const float *proj, int dim, int k, const int32_t *sel,
                                                                const float *prob, const float *db, int db_stride,
                                                                float *x) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int64_t t = blockIdx.y;
    if (i >= dim) return;
    float acc = 0.0f;
    for (int r = 0; r < k; r++) {
        const int64_t p = t * k + r;
        float v = proj[p * dim + i];
        if (db) v = v + db[(size_t)sel[p] * db_stride + i];
        acc += v * prob[p];
    }
    x[t * dim + i] += acc;
}

// The routed expert product: for every (token, slot) pair p = t k + r routed
// to expert e = sel[p], row r of e's MXFP4 matrix times the pair's activation.
struct MxExpArgs {
    const uint8_t *w[2];  // expert tensors: expert e's row r at w + e*exp_stride + r*row_stride
    float *y[2];          // [T*k][ldy]
    int64_t row_stride, exp_stride;
    int32_t rows, K, n_pairs, k;
    const float *x;  // the activation of pair p: x + (x_pair ? p : p / k) * ldx
    int64_t ldx, ldy;
    int32_t x_pair;
    const int32_t *sel;  // [n_pairs]
    int32_t n_exp;
};

// For every expert, the pairs routed to it in pair order (lists[e * cap ..]),
// their count, and the pair tiles of all experts.  For the serial product
// tiles[0] of them, tiles[1 + i] = e | (first pair / MXM_PAIRS) << 8: tiles of
// more than MXM_PAIRS / 2 pairs come first (they take twice the time of the
// others, and the last to start should be the short ones), each kind in expert
// order.  For the opt-in one (OFFSETS) tiles[e] = the tiles of MXO_PAIRS before
// expert e's, tiles[n_exp] = all.  One workgroup of up to 16 waves, each with a
// contiguous share of the pairs: it counts its pairs per expert, then writes its
// hits after the earlier waves'.  The lanes of 64 pairs that share an expert
// come from six ballots, one per bit of its number (a ballot per expert took 27
// us for 4004 pairs over 32 experts, with every step of the tile lists spilled;
// now 7.8).  Pairs that name no expert are in no list.
#define MXE_MAX_PAIRS 1024  // a token routes to an expert at most once: pairs per expert <= T
#define MXM_PAIRS 64  // pairs per tile of the serial product
#define MXO_PAIRS 32  // ... and of the opt-in one
#define MXM_ROWS 128
#define MXE_MAX_TILES (8 * MXE_MAX_PAIRS / MXM_PAIRS + 64)  // top_k <= 8, n_exp <= 64
// The lanes of the wave whose se is this lane's (0 where it names no expert).
__device__ __forceinline__ unsigned long long same_expert_lanes(int se, int n_exp) {
    const bool ok = (unsigned)se < (unsigned)n_exp;
    unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const bool bit = (se >> i) & 1;
        const unsigned long long set = __builtin_amdgcn_ballot_w64(bit);
        m &= bit ? set : ~set;
    }
    return ok ? m : 0ull;
}

// The tiles of PER pairs of the wave's experts, lane e's tot pairs being expert
// e's: n_long tiles more than half full, n_short (0 or 1) others, and how many
// there are of both up to and including this expert (below 2^15) and in all.
struct PairTiles {
    int full, n_long, n_short, long_upto, short_upto, long_all, short_all;
};
template <int PER>
__device__ __forceinline__ PairTiles pair_tiles(int tot, int lane) {
    PairTiles t;
    const int rem = tot % PER;
    t.full = tot / PER;
    t.n_long = t.full + (rem > PER / 2 ? 1 : 0);
    t.n_short = rem > 0 && rem <= PER / 2 ? 1 : 0;
    int upto = t.n_long << 16 | t.n_short;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, 64);
        upto += lane >= o ? v : 0;
    }
    const int all = __builtin_amdgcn_readlane(upto, 63);
    t.long_upto = upto >> 16;
    t.short_upto = upto & 0xFFFF;
    t.long_all = all >> 16;
    t.short_all = all & 0xFFFF;
    return t;
}

template <bool OFFSETS>
__global__ __launch_bounds__(1024) void moe_expert_lists_kernel(const int32_t *sel, int n_pairs, int n_exp, int cap,
                                                                 int32_t *lists, int32_t *counts, int32_t *tiles) {
    __shared__ int32_t s_cnt[16][64], s_at[16][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6, per = ((n_pairs + nw - 1) / nw + 63) / 64 * 64;
    const int pa = min(n_pairs, wave * per), pb = min(n_pairs, pa + per);
    // the first 64 pairs' experts stay in a register for the second pass
    const int first = pa + lane < pb ? sel[pa + lane] : -1;
    s_cnt[wave][lane] = 0;
    __syncthreads();
    for (int base = pa; base < pb; base += 64) {
        const int se = base == pa ? first : base + lane < pb ? sel[base + lane] : -1;
        const unsigned long long m = same_expert_lanes(se, n_exp);
        if (m != 0 && (m & ((1ull << lane) - 1ull)) == 0) atomicAdd(&s_cnt[wave][se], __builtin_popcountll(m));
    }
    __syncthreads();
    int off = 0, tot = 0;  // lane e: pairs of expert e in the earlier waves, in all waves
    for (int w = 0; w < nw; w++) {
        const int c = s_cnt[w][lane];
        off += w < wave ? c : 0;
        tot += c;
    }
    s_at[wave][lane] = off;
    __syncthreads();
    for (int base = pa; base < pb; base += 64) {
        const int se = base == pa ? first : base + lane < pb ? sel[base + lane] : -1;
        const unsigned long long m = same_expert_lanes(se, n_exp);
        const int before = __builtin_popcountll(m & ((1ull << lane) - 1ull));
        int at = 0;  // the first lane of each expert takes the places of all of them
        if (m != 0 && before == 0) at = atomicAdd(&s_at[wave][se], __builtin_popcountll(m));
        at = __shfl(at, m != 0 ? __builtin_ctzll(m) : lane, 64) + before;
        if (m != 0 && at < cap) lists[(size_t)se * cap + at] = base + lane;
    }
    if (wave == 0) {
        tot = lane < n_exp ? min(tot, cap) : 0;
        if (lane < n_exp) counts[lane] = tot;
        const PairTiles t = pair_tiles<OFFSETS ? MXO_PAIRS : MXM_PAIRS>(tot, lane);
        if (OFFSETS) {
            if (lane < n_exp) tiles[lane + 1] = t.long_upto + t.short_upto;
            if (lane == 0) tiles[0] = 0;
            return;
        }
        const int l0 = t.long_upto - t.n_long, s0 = t.long_all + t.short_upto - t.n_short;
        for (int i = 0; i < t.n_long; i++) tiles[1 + l0 + i] = lane | i << 8;
        if (t.n_short) tiles[1 + s0] = lane | t.full << 8;
        if (lane == 0) tiles[0] = t.long_all + t.short_all;
    }
}

// The same for one workgroup of the serial product without the list kernel:
// pair tile number `tile` of at most MXE_OWN_PAIRS pairs.  Fills s_pair and
// returns the tile's pairs (0: there is no such tile) and its expert.  Up to 64
// pairs every wave sees them all, and tile i is the expert of the i-th pair
// that is its expert's first; beyond, four waves with a quarter of the pairs in
// registers each count and rank as the list kernel does (0.5 us more).
#define MXE_OWN_PAIRS 1024
__device__ __forceinline__ int own_pair_tile(const int32_t *sel, int n_pairs, int n_exp, int tile, int32_t (*s_cnt)[64],
                                             int32_t *s_pair, int &expert) {
    constexpr int G = MXE_OWN_PAIRS / 256;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (n_pairs <= 64) {
        const int mine = lane < n_pairs ? sel[lane] : -1;
        const unsigned long long m = same_expert_lanes(mine, n_exp);
        const bool first = m != 0 && (m & below) == 0;
        const unsigned long long firsts = __builtin_amdgcn_ballot_w64(first);
        const unsigned long long at = __builtin_amdgcn_ballot_w64(first && __builtin_popcountll(firsts & below) == tile);
        if (at == 0) return 0;
        expert = __builtin_amdgcn_readlane(mine, __builtin_ctzll(at));
        const bool hit = mine == expert;
        const unsigned long long hits = __builtin_amdgcn_ballot_w64(hit);
        if (wave == 0 && hit) s_pair[__builtin_popcountll(hits & below)] = lane;
        return __builtin_popcountll(hits);
    }
    const int groups = (n_pairs + 255) / 256, pa = wave * groups * 64;
    int se[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int p = pa + 64 * g + lane;
        se[g] = g < groups && p < n_pairs ? sel[p] : -1;
    }
    s_cnt[wave][lane] = 0;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) {
        if (g >= groups) break;  // uniform
        const unsigned long long m = same_expert_lanes(se[g], n_exp);
        if (m != 0 && (m & below) == 0) atomicAdd(&s_cnt[wave][se[g]], __builtin_popcountll(m));
    }
    __syncthreads();
    int off = 0, tot = 0;  // lane e: pairs of expert e in the earlier waves, in all waves
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const int c = s_cnt[w][lane];
        off += w < wave ? c : 0;
        tot += c;
    }
    const PairTiles t = pair_tiles<MXM_PAIRS>(tot, lane);
    if (tile >= t.long_all + t.short_all) return 0;
    int e, p0;
    if (tile < t.long_all) {
        e = __builtin_ctzll(__builtin_amdgcn_ballot_w64(t.long_upto > tile));
        p0 = (tile - __builtin_amdgcn_readlane(t.long_upto - t.n_long, e)) * MXM_PAIRS;
    } else {
        e = __builtin_ctzll(__builtin_amdgcn_ballot_w64(t.short_upto > tile - t.long_all));
        p0 = __builtin_amdgcn_readlane(t.full, e) * MXM_PAIRS;
    }
    int at = __builtin_amdgcn_readlane(off, e) - p0;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const bool hit = se[g] == e;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(hit);
        const int i = at + __builtin_popcountll(m & below);
        if (hit && i >= 0 && i < MXM_PAIRS) s_pair[i] = pa + 64 * g + lane;
        at += __builtin_popcountll(m);
    }
    expert = e;
    return min(MXM_PAIRS, __builtin_amdgcn_readlane(tot, e) - p0);
}

// y[mat] row p for one (128-row tile, 64-pair tile of one expert, matrix).
// grid (ceil(rows / 128), an upper bound of the pair tiles, n_mats);
// workgroups past the last tile return.  Wave w owns rows row0 + 32 w ..
// + 31 and the tile's pairs in one or two groups of 32.
//
// Every sum is dot_mxfp4_f32_scalar's running sum, sum = sum + (w x) per element in
// order, bit for bit, on the matrix cores.  v_mfma_f32_32x32x2_f32 is a chain
// of two fused multiply-adds in k order, each rounded (checked on the device
// over normal, subnormal and mixed magnitudes), so a step of the chain with an
// exact product is the reference's step.  The product of x and a weight with
// magnitude 0.5, 1, 2 or 4 is exact; for 1.5, 3 and 6 the reference's rounded
// w x is (w / 3) RN(3 x), an exact product again.  So an element takes both k
// slots, (w1, x) and (w3, RN(3 x)), with w1 or w3 zero, and a zero product
// leaves the sum as it is: the sum starts at +0 and is never -0.  Lane half h
// = lane / 32 is k slot h: it holds w1 or w3 of row n = lane % 32 and x or
// RN(3 x) of pair n.  Scaling by w's power of two is exact while nothing
// leaves the normal range: a block whose |x| are 0 or in [2^-84, 2^80) and
// whose scales are within 2^-40 .. 2^40 qualifies (products stay above 2^-126
// and below 2^126); any other (zero, huge or non-finite values, scale bytes 0
// and 255 among them) takes the element-by-element sums on the VALU.
//
// The bound is the matrix cores, 64 clocks per 32 rows x 32 pairs x element
// (78 TFLOP/s of the reference's products), and an f32 MFMA leaves the VALU no
// room: a chain of 32x32x2 MFMAs takes 64 clocks each, 122 with twelve adds and
// multiplies after each one, interleaved or not.  Hence the 32x32 shape (half
// the operands per product of 16x16; 16-pair groups, 64 rows per workgroup and
// the factor 3 in the loop took 1504 us for 1024 pairs of 11520 x 2880, 57% of
// the bound), RN(3 x) computed once per workgroup into a plane of its own, and
// the code lookup on four nibbles per v_perm.  Weights come from a
// double-buffered LDS chunk of 8 blocks (rows of 136 bytes: 32 rows of a dword
// read are on distinct banks), the activations from two double-buffered planes
// (pitch 68 floats, 16-byte reads); both are loaded through registers one chunk
// or barrier ahead, 71 KB of LDS and two workgroups per CU.  A tile of up to 32
// pairs runs two blocks between barriers in the room of the second group's
// activations: where the grid leaves CUs idle a workgroup's time per block is
// what counts, 1.5 us with one block per barrier, the decode after the MFMAs and
// the range check as 24 compares, now 1.27 (0.85 of it MFMAs).
//
// Measured, us per call, against eight VALU sums per wave (x by scalar loads,
// 64-row workgroups): 1024 pairs of 11520 x 2880 1197 (57 TFLOP/s, 0.72 of the
// bound) : 11733; 1000 pairs over 32 experts of 2880 x 2880 (31 per expert:
// half-filled tiles) 499 : 898; 12 pairs 131 : 245; 6 pairs of 720 x 2880 126 :
// 136; 12 pairs of 96 x 96 19 : 19.  Over 288 shapes of 6 to 32 experts, 6 to
// 1000 pairs, 96 to 2880 rows and columns it is slower, by 3%, only where the
// tiles barely exceed the CUs and hold a pair or two each (264 workgroups: 224 :
// 216).  The 4004 gate/up pairs of a 1001-token gpt-oss-20b chunk take 2.5 ms
// (53 TFLOP/s), 6.9 with the VALU sums.
#define MXM_C 8  // weight blocks per LDS chunk
template <int PT>
__device__ __forceinline__ void mxfp4_experts_tile(const MxExpArgs &A, const uint8_t *w, float *y, int row0, int np,
                                                   uint2 *s_b, float *s_x, uint32_t *s_bad, const int32_t *s_pair) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef float v16f __attribute__((ext_vector_type(16)));
    constexpr int UB = 3 - PT;                      // blocks between barriers
    constexpr int XP = 68, XN = MXM_PAIRS * XP;     // row pitch and buffer size of s_x, in floats
    constexpr int WP = MXM_C * 17, WN = MXM_ROWS * 17;  // row bytes and buffer size (8-byte pieces) of s_b
    constexpr int NW = 32;                          // MFMAs per block and pair group
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int nb = A.K >> 5;
    // activations of UB blocks: thread t stages float4 t % 8 for rows t / 8 + 32 j
    // of s_x, row 32 j + i being pair 32 j + i (PT = 2) or block j of pair i
    const int c4 = tid & 7, pr0 = tid >> 3, nu = (nb + UB - 1) / UB;
    const float *xr[PT];
#pragma unroll
    for (int j = 0; j < PT; j++) {
        const int p = s_pair[min(pr0 + 32 * j, np - 1)];
        xr[j] = A.x + (A.x_pair ? (int64_t)p : (int64_t)(p / A.k)) * A.ldx + 4 * c4;
    }
    v4f xs[2];
    auto load_x = [&](int u) {
#pragma unroll
        for (int j = 0; j < 2; j++)
            __builtin_memcpy(&xs[j], PT == 2 ? xr[PT == 2 ? j : 0] + 32 * u : xr[0] + 32 * min(2 * u + j, nb - 1), 16);
    };
    auto store_x = [&](int u) {
        // the largest magnitude's bits, and the smallest's that is not 0, less 1
        uint32_t hi = 0, lo = 0xFFFFFFFFu;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float *r = s_x + (u & 1) * XN + (pr0 + 32 * j) * XP;
            const v4f v = xs[j];
            *(v4f *)(r + 4 * c4) = v;
            *(v4f *)(r + 32 + 4 * c4) = v * 3.0f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t f = __float_as_uint(v[i]) & 0x7FFFFFFFu;  // (a bit_cast of v[i] reads v[0])
                hi = max(hi, f);
                lo = min(lo, f - 1u);
            }
        }
        const bool bad = hi >= __builtin_bit_cast(uint32_t, 0x1p80f) || lo < __builtin_bit_cast(uint32_t, 0x1p-84f) - 1u;
        const uint32_t any = __builtin_amdgcn_ballot_w64(bad) != 0 ? 1u : 0u;
        if (lane == 0) s_bad[4 * (u & 1) + wave] = any;
    };
    // weights: piece f = 256 i + t of a chunk is row f / 17, bytes 8 (f % 17)
    constexpr int NP = (WN + 255) / 256;
    uint2 wg[NP];
    auto load_w = [&](int c) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int f = min(256 * i + tid, WN - 1), r = f / 17, p = f - 17 * r;
            const int rr = min(row0 + r, A.rows - 1);
            const int64_t o = min((int64_t)(WP * c + 8 * p), A.row_stride - 8);
            wg[i] = ld8(w + (int64_t)rr * A.row_stride + o);
        }
    };
    auto store_w = [&](int c) {
        uint2 *d = s_b + (c & 1) * WN;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (256 * i + 256 <= WN || 256 * i + tid < WN) d[256 * i + tid] = wg[i];
    };
    // the weights k slot h takes of the eight magnitudes: 0.5, 1, 2 and 4, or
    // a third of 1.5, 3 and 6
    const uint32_t tlo = h ? 0x01000000u : 0x00020100u, thi = h ? 0x04000200u : 0x00060004u;
    const uint8_t *rowb0 = (const uint8_t *)s_b + (32 * wave + n) * WP;
    // block b's weights of this lane's k slot; returns whether a scale needs
    // the element path
    auto decode = [&](int b, float (&wv)[NW]) -> bool {
        const int j = b & (MXM_C - 1);
        // the block's 17 bytes from byte 17 j of the row, five aligned dwords
        const uint32_t *wp = (const uint32_t *)(rowb0 + ((b / MXM_C) & 1) * (WN * 8) + ((17 * j) & ~3));
        const uint32_t sb = (uint32_t)j & 3u;  // 17 j mod 4
        uint32_t dw[5], wd[4];
#pragma unroll
        for (int i = 0; i < 5; i++) dw[i] = wp[i];
#pragma unroll
        for (int i = 0; i < 4; i++) wd[i] = __builtin_amdgcn_alignbyte(dw[i + 1], dw[i], sb);
        const uint32_t ex = (dw[4] >> (8u * sb)) & 0xFFu;
        const float sc = __builtin_bit_cast(float, ex << 23);  // 2^(ex - 127) where it is used: 0 < ex < 255
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t lo = __builtin_amdgcn_perm(thi, tlo, wd[q] & 0x07070707u);
            const uint32_t hi = __builtin_amdgcn_perm(thi, tlo, (wd[q] >> 4) & 0x07070707u);
            const uint32_t u = (lo | (hi << 4)) | (wd[q] & 0x88888888u);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const fp4x2_f32 p = fp4x2_scaled(u, sc, i);
                wv[8 * q + 2 * i] = p.x;
                wv[8 * q + 2 * i + 1] = p.y;
            }
        }
        return ex - 87u > 80u;
    };
    v16f acc[PT];
#pragma unroll
    for (int g = 0; g < PT; g++) acc[g] = v16f{};
    // block b from the LDS bytes, element by element: C element i of lane
    // (n, h) is (pair 8 (i / 4) + 4 h + i % 4, row n)
    auto slow_block = [&](int b) {
        const int j = b & (MXM_C - 1);
        const uint8_t *blk = rowb0 + ((b / MXM_C) & 1) * (WN * 8) + 17 * j;
        const float sc = mxfp4_scale(blk[16]);
        const float *xc = s_x + ((b / UB) & 1) * XN + (32 * (b % UB) + 4 * h) * XP;
#pragma unroll 1
        for (int e = 0; e < 32; e++) {
            const uint32_t byte = blk[e >> 1];
            const float wv = mxfp4_nibble((e & 1) ? byte >> 4 : byte & 0xFu) * sc;
#pragma unroll
            for (int g = 0; g < PT; g++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    acc[g][i] += wv * xc[(32 * g + 8 * (i >> 2) + (i & 3)) * XP + e];
        }
    };
    load_w(0);
    load_x(0);
    store_w(0);
    store_x(0);
    load_x(min(1, nu - 1));
    float wa[NW], wb[NW];
    const float *xb0 = s_x + n * XP + 32 * h;
    __syncthreads();  // the first chunk is in LDS
    bool odd = __builtin_amdgcn_ballot_w64(decode(0, wa)) != 0;
    v4f xv[NW / 4][2];
    // block b, its weights in cur, its activations in xv; the next block's
    // weights go to nxt, decoded while the MFMAs run
    auto block = [&](int b, auto half, bool slow, const float (&cur)[NW], float (&nxt)[NW]) {
        constexpr int O = decltype(half)::value;  // b % 2
        bool bad;
        if (slow) {
            slow_block(b);
            bad = decode(min(b + 1, nb - 1), nxt);
        } else {
            bad = decode(min(b + 1, nb - 1), nxt);
#pragma unroll
            for (int i = 0; i < NW; i++)
#pragma unroll
                for (int g = 0; g < PT; g++)
                    acc[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i >> 2][PT == 2 ? g : O][i & 3], cur[i], acc[g],
                                                                  0, 0, 0);
        }
        odd = __builtin_amdgcn_ballot_w64(bad) != 0;
    };
    // unit u of UB blocks: returns whether its activations need the element path
    auto enter = [&](int u) -> bool {
        __syncthreads();  // unit u is in LDS; unit u - 1's reads are done
        if (u + 1 < nu) store_x(u + 1);
        if (u + 2 < nu) load_x(u + 2);
        // the next weight chunk, one barrier before the decode ahead reads it
        const int c = UB * u / MXM_C, j = UB * u & (MXM_C - 1);
        if (MXM_C * (c + 1) < nb) {
            if (j == UB) load_w(c + 1);
            if (j == MXM_C - 2 * UB) store_w(c + 1);
        }
        const float *xc = xb0 + (u & 1) * XN;
#pragma unroll
        for (int q = 0; q < NW / 4; q++)
#pragma unroll
            for (int g = 0; g < 2; g++) xv[q][g] = *(const v4f *)(xc + 32 * g * XP + 4 * q);
        const uint4 b4 = *(const uint4 *)(s_bad + 4 * (u & 1));
        return __builtin_amdgcn_readfirstlane(b4.x | b4.y | b4.z | b4.w) != 0;
    };
    for (int b = 0; b < nb; b += 2) {
        bool xbad = enter(b / UB);
        block(b, std::integral_constant<int, 0>(), odd || xbad, wa, wb);
        if (b + 1 >= nb) break;
        if (UB == 1) xbad = enter(b + 1);
        block(b + 1, std::integral_constant<int, 1>(), odd || xbad, wb, wa);
    }
    const int row = row0 + 32 * wave + n;
    if (row >= A.rows) return;
#pragma unroll
    for (int g = 0; g < PT; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int p = 32 * g + 8 * (i >> 2) + 4 * h + (i & 3);
            if (p < np) y[(int64_t)s_pair[p] * A.ldy + row] = acc[g][i];
        }
}

// lists null: every workgroup finds its own pairs (own_pair_tile).
__global__ __launch_bounds__(256, 2) void gemm_mxfp4_experts_kernel(MxExpArgs A, const int32_t *lists,
                                                                    const int32_t *counts, const int32_t *tiles,
                                                                    int cap) {
    __shared__ __align__(16) uint2 s_b[2 * MXM_ROWS * 17];
    __shared__ __align__(16) float s_x[2 * MXM_PAIRS * 68];
    __shared__ __align__(16) uint32_t s_bad[8];
    __shared__ int32_t s_pair[MXM_PAIRS], s_cnt[4][64];
    const int mat = blockIdx.z;
    int e, np;
    if (lists) {
        if ((int)blockIdx.y >= tiles[0]) return;  // uniform
        const int tile = tiles[1 + blockIdx.y], p0 = (tile >> 8) * MXM_PAIRS;
        e = tile & 0xFF;
        np = min(MXM_PAIRS, counts[e] - p0);
        if ((int)threadIdx.x < np) s_pair[threadIdx.x] = lists[(size_t)e * cap + p0 + threadIdx.x];
    } else {
        np = own_pair_tile(A.sel, A.n_pairs, A.n_exp, blockIdx.y, s_cnt, s_pair, e);
        if (np == 0) return;  // uniform
    }
    __syncthreads();
    const uint8_t *w = A.w[mat] + (int64_t)e * A.exp_stride;
    float *y = A.y[mat];
    const int row0 = blockIdx.x * MXM_ROWS;
    if (np > 32)
        mxfp4_experts_tile<2>(A, w, y, row0, np, s_b, s_x, s_bad, s_pair);
    else
        mxfp4_experts_tile<1>(A, w, y, row0, np, s_b, s_x, s_bad, s_pair);
}

// ---- opt-in expert product on the matrix cores ------------------------------
// Sums of unrounded products in the matrix cores' own order: not bit-exact, and
// off unless rusty_hip_set_expert_mfma(1) selects it.  Its inputs keep the
// reference's precision: the weights lut[n] * 2^(e-127) are exact in f32 and
// the activations are the f32 rows; only the order and rounding of the f32
// additions of the K products differ (v_mfma_f32_32x32x2_f32).
//
// y[mat] row p = expert rows times pair p's activation for one (128-row tile,
// 32-pair tile of one expert, matrix): grid (ceil(rows / 128), an upper bound
// of the pair tiles, n_mats); workgroups past tile0[n_exp] return.  Wave w
// owns rows row0 + 32 w + (lane % 32); per 32-element block, 16 MFMAs
// 32x32x2: MFMA i takes element 16 h + i (h = lane / 32) of the block from
// both operands, A = the pair's activation (m = pair), B = the weight (n =
// row), so lane h decodes bytes 8h..8h+7 of its row's block (element 2b + 1
// is the high nibble of byte b).  The weights arrive in 16-block chunks of
// 272 bytes per row by coalesced direct loads into a double-buffered LDS
// chunk; each lane then reads its row's chunk into registers (17 reads, an
// odd number of 16-byte units per row: conflict-free); the activations come
// from global memory one block ahead.
//
// Bound by the latency of a workgroup's K loop until the grid passes two
// workgroups per CU: hence 32 pairs per tile, a second tile going to a second
// CU, and one barrier per 16 blocks.  Measured, us per call, against this
// product in the serial kernel's tiles (64 pairs, activations in LDS, a barrier
// per block): 6 experts x 720 x 2880, 256 pairs 73 : 137, 1000 pairs 84 : 141;
// 32 experts x 2880 x 2880, 64 pairs 171 : 212, 1000 pairs 277 : 306; prefill of
// 1001 tokens, 4 gpt-oss-20b layers, 18.9 ms (26.8 with the serial sums).  A
// workgroup looks its expert up by walking the offsets: with the tile list
// instead all start at once, the 736 workgroups of 32 experts x 2880 rows end
// together too, and the second round lands two to a CU: 215 : 172.
__global__ __launch_bounds__(256) void gemm_mxfp4_experts_mfma_kernel(MxExpArgs A, const int32_t *lists,
                                                                      const int32_t *counts, const int32_t *tile0,
                                                                      int cap) {
    __shared__ __align__(16) uint4 s_b[2][MXM_ROWS * 17];
    __shared__ int32_t s_pair[MXO_PAIRS];
    typedef float v16f __attribute__((ext_vector_type(16)));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mat = blockIdx.z, gt = blockIdx.y;
    const int n_exp = A.n_exp;
    if (gt >= tile0[n_exp]) return;  // uniform
    int e = 0;
    while (e + 1 < n_exp && tile0[e + 1] <= gt) e++;
    const int p0 = (gt - tile0[e]) * MXO_PAIRS;
    const int np = min(MXO_PAIRS, counts[e] - p0);
    if (tid < MXO_PAIRS) s_pair[tid] = lists[(size_t)e * cap + p0 + min(tid, np - 1)];
    const int m = lane & 31, h = lane >> 5;
    const int row0 = blockIdx.x * MXM_ROWS, row = row0 + 32 * wave + m;
    const uint8_t *w = A.w[mat] + (int64_t)e * A.exp_stride;
    const int64_t stride = A.row_stride;
    const int nb = A.K >> 5, nch = (nb + MXF_C - 1) / MXF_C;
    // piece f = 256 i + tid of a chunk: row f / 17, bytes 16 (f % 17); the
    // 2176 pieces are 34 whole wave instructions, so a wave's instruction is
    // either all inside the chunk or skipped
    auto issue_chunk = [&](int c, int buf) {
#pragma unroll
        for (int i = 0; i < 9; i++) {
            if (256 * i + 64 * wave >= MXM_ROWS * 17) continue;  // uniform
            const int f = 256 * i + tid, r = f / 17, pc = f - 17 * r;
            const int rr = min(row0 + r, A.rows - 1);
            const int64_t o = min((int64_t)(MXF_C * 17 * c + 16 * pc), stride - 16);
            dma16(w + (int64_t)rr * stride + o, &s_b[buf][256 * i + 64 * wave]);
        }
    };
    issue_chunk(0, 0);
    __syncthreads();  // s_pair
    const int pair = s_pair[m];
    const float *xr = A.x + (A.x_pair ? (int64_t)pair : (int64_t)(pair / A.k)) * A.ldx + 16 * h;
    float4 xa[4], xb[4];
    auto load_x = [&](int b, float4 (&xv)[4]) {
        const float4 *p = (const float4 *)(xr + 32 * (int64_t)min(b, nb - 1));
#pragma unroll
        for (int q = 0; q < 4; q++) xv[q] = p[q];
    };
    load_x(0, xa);
    v16f acc = {};
    for (int c = 0; c < nch; c++) {
        RH_WAIT_VM(0);
        __syncthreads();  // chunk c landed from every wave; every read of chunk c - 1 done
        uint32_t wr[68];
        {
            const uint4 *rp = &s_b[c & 1][(32 * wave + m) * 17];
#pragma unroll
            for (int q = 0; q < 17; q++) {
                const uint4 v = rp[q];
                wr[4 * q] = v.x;
                wr[4 * q + 1] = v.y;
                wr[4 * q + 2] = v.z;
                wr[4 * q + 3] = v.w;
            }
        }
        // block j of the chunk with its activations in cur; the next block's
        // go to nxt (clamped past the end), then, late in the chunk, the next
        // chunk's weights are issued: a load issued after them would wait for
        // them too (loads retire in order), and only the next chunk's first
        // activations are
        auto block = [&](int j, const float4 (&cur)[4], float4 (&nxt)[4]) {
            const int b = MXF_C * c + j;
            if (b >= nb) return;  // uniform
            load_x(b + 1, nxt);
            if (j == MXF_C - 2 && c + 1 < nch) issue_chunk(c + 1, (c + 1) & 1);
            // bytes 17 j + 8 h .. + 7 and the scale byte 17 j + 16
            const int o0 = 17 * j, o1 = 17 * j + 8, os = 17 * j + 16;
            const uint32_t a0 = __builtin_amdgcn_alignbyte(wr[o0 / 4 + 1], wr[o0 / 4], o0 % 4);
            const uint32_t a1 = __builtin_amdgcn_alignbyte(wr[o0 / 4 + 2], wr[o0 / 4 + 1], o0 % 4);
            const uint32_t c0 = __builtin_amdgcn_alignbyte(wr[o1 / 4 + 1], wr[o1 / 4], o1 % 4);
            const uint32_t c1 = __builtin_amdgcn_alignbyte(wr[o1 / 4 + 2], wr[o1 / 4 + 1], o1 % 4);
            const uint32_t d0 = h ? c0 : a0, d1 = h ? c1 : a1;
            const uint32_t ex = (wr[os / 4] >> (8 * (os % 4))) & 0xFFu;
            const float sc = mxfp4_scale(ex);
            float wv[16];
            if (__builtin_amdgcn_ballot_w64(ex == 0u || ex == 255u) == 0) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const fp4x2_f32 lo = fp4x2_scaled(d0, sc, u), hi = fp4x2_scaled(d1, sc, u);
                    wv[2 * u] = lo.x;
                    wv[2 * u + 1] = lo.y;
                    wv[8 + 2 * u] = hi.x;
                    wv[9 + 2 * u] = hi.y;
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t b0 = (d0 >> (8 * u)) & 0xFFu, b1 = (d1 >> (8 * u)) & 0xFFu;
                    wv[2 * u] = mxfp4_nibble(b0 & 0xFu) * sc;
                    wv[2 * u + 1] = mxfp4_nibble(b0 >> 4) * sc;
                    wv[8 + 2 * u] = mxfp4_nibble(b1 & 0xFu) * sc;
                    wv[9 + 2 * u] = mxfp4_nibble(b1 >> 4) * sc;
                }
            }
            const float xs[16] = {cur[0].x, cur[0].y, cur[0].z, cur[0].w, cur[1].x, cur[1].y, cur[1].z, cur[1].w,
                                  cur[2].x, cur[2].y, cur[2].z, cur[2].w, cur[3].x, cur[3].y, cur[3].z, cur[3].w};
#pragma unroll
            for (int i = 0; i < 16; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[i], wv[i], acc, 0, 0, 0);
        };
#pragma unroll
        for (int j = 0; j < MXF_C; j += 2) {
            block(j, xa, xb);
            block(j + 1, xb, xa);
        }
    }
    if (row >= A.rows) return;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int mi = 8 * (i >> 2) + 4 * h + (i & 3);
        if (mi < np) A.y[mat][(int64_t)s_pair[mi] * A.ldy + row] = acc[i];
    }
}

// K/V rows between a ring cache and the linear buffer of a batched ring
// prefill: gather lin[r] = ring[(p0 + r) % S] for r < n rows; scatter
// ring[(p0 + r) % S] = lin[off + r].  grid (ceil(width/256), n, 2 (K, V)).
__global__ __launch_bounds__(256) void kv_ring_copy_kernel(float *kring, float *vring, float *klin, float *vlin,
                                                           int kw, int vw, int p0, int S, int off, int to_ring) {
    const int r = blockIdx.y, which = blockIdx.z, c = blockIdx.x * 256 + threadIdx.x;
    const int w = which ? vw : kw;
    if (c >= w) return;
    float *ring = which ? vring : kring;
    float *lin = which ? vlin : klin;
    const int64_t slot = (p0 + r) % S;
    if (to_ring)
        ring[slot * w + c] = lin[(int64_t)(off + r) * w + c];
    else
        lin[(int64_t)r * w + c] = ring[slot * w + c];
}

}  // namespace rh
