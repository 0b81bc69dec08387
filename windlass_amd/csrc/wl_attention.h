// wl_attention.h - host interface of the prompt rows' attention on the matrix cores.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wl {

// Whether it takes T consecutive rows of one sequence (cache rows 16-byte aligned).
bool attention_tiles_applies(int T, int hd);
// Floats of scratch for rows that attend to at most max_n positions (pos0 + T).
int64_t attention_tiles_scratch_floats(int T, int heads, int kv_heads, int hd, int max_n);
// out [T][ldo] = attention of rows q [T][ldq] at positions pos0.. over the caches K, V
// [positions][kv_dim]; out rows 16-byte aligned.
hipError_t attention_tiles_launch(const float *q, int64_t ldq, int T, const uint16_t *K, const uint16_t *V, int kv_dim,
                                  int heads, int kv_heads, int hd, int pos0, float scale, float *part, float *out,
                                  int64_t ldo, hipStream_t st);

}  // namespace wl
