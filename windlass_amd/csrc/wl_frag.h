// wl_frag.h - the orders in which a prompt's activations reach the bf16 matrix cores: 16-byte
// pieces of 8 consecutive columns of one token, contiguous in the order a wave loads them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wl {

// Tokens whose pieces lie together, and bytes of T tokens x cols.
__host__ __device__ inline int frag_tokens(int ord) { return ord == 2 ? 32 : 16; }
__host__ __device__ inline int64_t frag_bytes(int T, int cols, int ord) {
  const int n = frag_tokens(ord);
  return (int64_t)((T + n - 1) / n) * n * cols * 2;
}

// The place of x[t][k .. k+7] (k % 8 == 0) of rows of cols columns, in pieces.
//   0, 1: v_mfma_f32_16x16x32_bf16, 16 tokens x 256 columns as 8 chunks of 64 lanes; lane 16 q + t
//         has 64 of the 256 columns: 128 hh + 32 g + 16 ih + (0..15) with q = 2 hh + ih (0), or
//         64 q + (0..63) (1), 8 a chunk
//   2:    v_mfma_f32_32x32x16_bf16, 32 tokens x 32 columns as 2 halves of 64 lanes
__host__ __device__ inline int64_t frag_at(int t, int k, int cols, int ord) {
  if (ord == 2)
    return (((int64_t)(t >> 5) * (cols >> 5) + (k >> 5)) * 2 + ((k >> 4) & 1)) * 64 + 32 * ((k >> 3) & 1) + (t & 31);
  const int q = ord ? (k >> 6) & 3 : 2 * ((k >> 7) & 1) + ((k >> 4) & 1);
  const int m = ord ? (k >> 3) & 7 : 2 * ((k >> 5) & 3) + ((k >> 3) & 1);
  return (((int64_t)(t >> 4) * (cols >> 8) + (k >> 8)) * 8 + m) * 64 + 16 * q + (t & 15);
}

}  // namespace wl
