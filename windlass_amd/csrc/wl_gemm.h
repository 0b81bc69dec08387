// wl_gemm.h - host-side interface of the prefill GEMM (bf16 MFMA, fp32 accumulation).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wl {

bool gemm_supports(int type);

// K-chunks of a launch (1 when the output tiles alone fill the device).
int gemm_chunks(int type, int rows, int cols, int T, int num_cu);
// Bytes of scratch gemm_launch needs: x as bf16, then the chunk partials when K is split.
int64_t gemm_scratch_bytes(int type, int rows, int cols, int T, int num_cu);

// y[t * ldy + r] = sum_k W[r][k] * x[t][k] for T rows of x (x is [T][cols] fp32), W rows x cols
// raw blocks of `type`. The operands enter the matrix cores as bf16 (weights decoded exactly in
// fp32, then rounded to nearest even; x rounded the same way into `scratch`); products and sums
// are fp32. A split K adds the chunk partials in chunk order, so results are deterministic.
hipError_t gemm_launch(int type, const uint8_t *w, int64_t row_bytes, int rows, int cols, const float *x, int T,
                       float *y, int ldy, void *scratch, int num_cu, hipStream_t st);

// Prompts of more than 128 tokens over Q8_0, Q4_K, Q5_K, Q6_K and IQ4_XS rows (wl_gemm_tall.hip): x (or
// silu(g) * u) as bf16 pieces in order 2 of wl_frag.h, then up to three matrices on them in one
// launch (y, or y += result * rs), with tall_part_bytes of scratch: the planes of the best K split, or,
// where those pass `limit` and the planes of one tile a CU do not, of the best split within it.
bool gemm_tall_applies(int type, int T, int64_t cols);
constexpr int TALL_MAX_MATS = 3;
// Columns at most: a wave's four token blocks of them are 1 GiB of pieces, within 32-bit offsets.
constexpr int64_t TALL_MAX_COLS = 1 << 22;
struct TallMat {
  const uint8_t *w;
  int64_t row_bytes;
  int rows, type;
  float *y;
  int64_t ldy;
};
hipError_t tall_frag_launch(const float *x, int T, int cols, void *xf, hipStream_t st);
hipError_t tall_silu_frag_launch(const float *g, const float *u, int T, int cols, void *xf, hipStream_t st);
int64_t tall_part_bytes(const TallMat *mats, int n, int cols, int T, int num_cu, int64_t limit);
hipError_t tall_matmul_launch(const TallMat *mats, int n, int cols, const void *xf, int T, bool add, float rs,
                              void *part, int64_t part_bytes, int num_cu, hipStream_t st);

}  // namespace wl
