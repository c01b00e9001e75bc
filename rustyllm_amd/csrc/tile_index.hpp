// Index arithmetic of the batched products that a host program can run too:
// the tests walk every lane of every tile through it.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define RH_HOST_DEVICE __host__ __device__
#else
#define RH_HOST_DEVICE
#endif

namespace rh {

// Rows that the quantized activations of T tokens are laid out in: whole
// 64-token tiles.  The K-quant products load whole tiles of quants and do not
// ask where the batch ends (their loads' scalar offset is not part of a raw
// buffer load's range check, so the buffer's extent cannot ask either); rows
// past T hold anything, and nothing computed from them is stored.
RH_HOST_DEVICE constexpr int64_t batch_rows(int64_t T) { return (T + 63) / 64 * 64; }

// Piece j of thread tid (256 threads) of a token tile's block b is the 16
// bytes at gemm_x_lane(tid, K) + gemm_x_step(j, b, K) from the tile's first
// token (K bytes per token): part tid % 16 of token tid / 16 + 16 j.
RH_HOST_DEVICE constexpr int gemm_x_lane(int tid, int K) { return (tid >> 4) * K + 16 * (tid & 15); }
RH_HOST_DEVICE constexpr int gemm_x_step(int j, int b, int K) { return 16 * j * K + 256 * b; }

}  // namespace rh
