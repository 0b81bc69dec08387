// wl_gemm_short.h - prompts of 9 to 128 tokens over Q8_0, Q4_K, Q5_K, Q6_K and IQ4_XS
// rows on the bf16 matrix cores (the batch branch of Transformer.MatMul,
// src/Transformer.cs:526-536): host interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wl_frag.h"

namespace wl {

constexpr int SHORT_MAX_MATS = 3;

// One matrix of a launch: y[t * ldy + r] = sum_k W[r][k] x[t][k] (added into y times rs with the
// launch's add).
struct ShortMat {
  const uint8_t *w;
  int64_t row_bytes;
  int rows, type;
  float *y;
  int64_t ldy;
};

bool short_type(int type);
// Whether a prompt of T tokens over rows of this type and length takes this kernel.
bool short_applies(int type, int T, int64_t cols);

// The order of x (wl_frag.h) that this type's operands have: 0 or 1.
inline int short_order(int type) { return type == 8 || type == 23; }

// fp32 x [T][cols] -> bf16 pieces (round to nearest even) in that order.
hipError_t short_frag_launch(const float *x, int T, int cols, int ord, void *xf, hipStream_t st);
// n matrices of one column count and order on the same x, in one launch.
hipError_t short_matmul_launch(const ShortMat *mats, int n, int cols, const void *xf, int T, bool add, float rs,
                               int num_cu, hipStream_t st);
// silu(gate x) * (up x) of two matrices of one type and shape (rows a multiple of 256), as the
// pieces hf (order hord) of the product that reads them.
hipError_t short_swiglu_launch(const ShortMat &gate, const ShortMat &up, int cols, const void *xf, int T, void *hf,
                               int hord, hipStream_t st);

}  // namespace wl
