// wl_attention.hip - attention of a prompt's rows on the matrix cores (head dims 64 and 128).
//
// What bounds it: scores and values are 4 T n HD flops per head on v_mfma_f32_32x32x16_f16, twice
// because the fp32 operands enter as two fp16 parts; at 2,048 tokens after 2,048 positions of a
// 32-head layer that is 206 GFLOP, about 130 us at this card's matrix rate, and the softmax's
// exponentials cost about half as much again on the VALU. The row-by-row kernel it replaces
// there (attention_rows_kernel: VALU products, exp in double) took 4,643 + 115 us; this one takes 343
// (600 TFLOP/s). 64 heads, 512 tokens: 245 -> 44 us; 32 heads, 45 tokens after 300: 31 -> 17 us.
// Root mean square error against float64: 0.4 to 0.93 of the row kernel's over 16 to 2,048 rows after 0
// to 3,000 positions with queries of deviation 0.3 to 30 (6.6e-8 against 7.4e-8 for 38 rows with 0.3).
//
// Arithmetic, at fp32's precision (Attention, src/Transformer.cs:351-393): the caches' fp16 keys
// and values are exact operands. A query row is scaled by a power of two and split into
// hi = fp16(q f), lo = fp16(q f - hi): 22 significant bits down to 2^-17 of the head's largest value,
// 2^-39 of that value below; exact products, fp32 sums. The probabilities are exp2 in fp32 of
// (score - running maximum) times the scale: the difference first, so that the argument's rounding
// is relative to the argument (a maximum scaled and rounded by itself, 14 up, left 1.6e-7 in flat
// softmaxes, and past scores of 2^26 no probability near 1). They enter the products as two fp16
// parts of 2^14 p: 22 bits down to 2^-16 of the largest, 2^-39 of the largest below. The denominator
// is summed in fp32 per 64 positions and in double across them.
//
// Layout. S^T = K Q^T puts a query in a lane column: lane l holds 16 of every 32 keys' scores of
// query l % 32, so the maximum takes one exchange with lane l ^ 32, and the probabilities are
// already the B operand of O^T = V^T P^T (the keys a half-wave holds, in the order its registers
// hold them; V is staged transposed in that order). A workgroup of four waves shares 64 keys and
// values in LDS per step; a wave owns 32 tokens of one query head, and the waves of a workgroup
// take (token block, head of the KV group) in turn, so a KV head's rows are read once per four.
//
// Infinities and NaN in the caches: a key or value only reaches the rows that attend to it. A
// step whose staged rows hold one takes slower branches: the parts' scores apart (inf times
// the low part is not added), and its non-finite values set to zero for the products and added to
// the rows that see them.
#include "wl_attention.h"
#include "wl_fmma_codec.h"

#pragma clang fp contract(off)

namespace wl {

typedef float ff16 __attribute__((ext_vector_type(16)));

constexpr int kAtK = 64;   // keys per step
constexpr int kAtQ = 32;   // tokens per wave
constexpr int kAtW = 4;    // waves per workgroup
constexpr float kAtUp = 0x1p14f;  // the probabilities' factor in their fp16 parts

__device__ __forceinline__ uint32_t pk_umax16(uint32_t a, uint32_t b) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, a), __builtin_bit_cast(us2, b)));
}
// the larger of acc and the halves' magnitudes; past 0x7bff in a half: an infinity or NaN
__device__ __forceinline__ void mag16(u32x4_t v, uint32_t &acc) {
  acc = pk_umax16(acc, v.x & 0x7fff7fffu);
  acc = pk_umax16(acc, v.y & 0x7fff7fffu);
  acc = pk_umax16(acc, v.z & 0x7fff7fffu);
  acc = pk_umax16(acc, v.w & 0x7fff7fffu);
}
__device__ __forceinline__ bool nonfinite16(uint32_t m) { return (m & 0x7fffu) > 0x7bffu || (m >> 16) > 0x7bffu; }
__device__ __forceinline__ uint32_t finite_pair(uint32_t v) {
  if ((v & 0x7c00u) == 0x7c00u) v &= 0xffff0000u;
  if ((v & 0x7c000000u) == 0x7c000000u) v &= 0xffffu;
  return v;
}

template <int HD>
__global__ __launch_bounds__(256, 2) void attention_tiles_kernel(const float *__restrict__ q, int64_t ldq,
                                                                const uint16_t *__restrict__ K,
                                                                const uint16_t *__restrict__ V, int kv_dim, int KH,
                                                                int G, int chunks, int nz, int T, int pos0,
                                                                float scale, int chunk, float *__restrict__ part,
                                                                float *__restrict__ out, int64_t ldo) {
  constexpr int NK = HD / 16, ND = HD / 32, U = HD / 8;  // key steps, value blocks, 16-byte pieces of a row
  constexpr int KS = HD + 8, VS = kAtK + 8;              // LDS row strides (halves): 16-byte reads hit every bank
  __shared__ __attribute__((aligned(16))) uint16_t ks[kAtK * KS];
  __shared__ __attribute__((aligned(16))) uint16_t vs[HD * VS];
  __shared__ int bads[2][kAtW];
  const int kvh = blockIdx.x % KH, c = blockIdx.x / KH % chunks, r = blockIdx.x / KH / chunks;
  // longest and shortest rows in turn: the workgroups that share a CU (the grid's halves) add up
  const int z = r < (nz + 1) / 2 ? nz - 1 - r : r - (nz + 1) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hf = lane >> 5, col = lane & 31;
  const int ntb = (T + kAtQ - 1) / kAtQ, NU = ntb * G;
  const int u = z * kAtW + wv, tb = u < NU ? u / G : ntb - 1, g = u < NU ? u % G : 0;
  const int ulast = z * kAtW + kAtW - 1 < NU ? z * kAtW + kAtW - 1 : NU - 1;
  const int tend = (ulast / G + 1) * kAtQ < T ? (ulast / G + 1) * kAtQ : T;
  const int nwg = pos0 + tend, k0 = c * chunk;  // positions the workgroup's rows read
  if (k0 >= nwg) return;                        // uniform over the workgroup
  const int kend = nwg < k0 + chunk ? nwg : k0 + chunk;
  const int t = tb * kAtQ + col < T ? tb * kAtQ + col : T - 1;
  const int lim = pos0 + t, limw = pos0 + tb * kAtQ;          // this row's last position; the wave's first row's
  const int nwave = pos0 + ((tb + 1) * kAtQ < T ? (tb + 1) * kAtQ : T);  // positions the wave's rows read
  const int h = kvh * G + g;

  // the query's parts, in operand order: k = 16 i + 8 hf + 0..7
  fh8 qh[NK], ql[NK];
  float c2;
  {
    const float *qp = q + (int64_t)t * ldq + (int64_t)h * HD + 8 * hf;
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NK; i++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float a = fabsf(qp[16 * i + j]);
        m = a < INFINITY ? fmaxf(m, a) : m;
      }
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    float f, inv;
    unit_scale(m, f, inv);
    // scores in units of log2: c2 > 0 (a negative scale negates the query)
    c2 = fmaxf(fabsf(scale) * 1.4426950408889634f * inv, 1.1754944e-38f);
    f = scale < 0.f ? -f : f;
    if (scale != scale) c2 = scale;
#pragma unroll
    for (int i = 0; i < NK; i++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float X = qp[16 * i + j] * f;
        const _Float16 a = (_Float16)X;
        qh[i][j] = a;
        ql[i][j] = (_Float16)(__builtin_isinf(X) ? 0.f : X - (float)a);
      }
  }
  ff16 O[ND];
#pragma unroll
  for (int d = 0; d < ND; d++)
#pragma unroll
    for (int i = 0; i < 16; i++) O[d][i] = 0.f;
  float M = -INFINITY;
  double L = 0.0;

  // staging: K pieces tid + 256 i (row / U, piece % U); V four rows 4 kg .. 4 kg + 3, piece dg
  const int kg = tid & 15, dg = tid >> 4;
  const uint16_t *Kb = K + (int64_t)kvh * HD, *Vb = V + (int64_t)kvh * HD;
  constexpr int KI = kAtK * U / 256;
  u32x4_t kr[KI], vr[4];
  auto fetch = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KI; i++) {
      const int e = tid + 256 * i;
      const int row = j0 + e / U < kend ? j0 + e / U : kend - 1;  // past the end: the last row again, masked
      kr[i] = *reinterpret_cast<const u32x4_t *>(Kb + (int64_t)row * kv_dim + 8 * (e % U));
    }
    if (dg < U) {
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int row = j0 + 4 * kg + b < kend ? j0 + 4 * kg + b : kend - 1;
        vr[b] = *reinterpret_cast<const u32x4_t *>(Vb + (int64_t)row * kv_dim + 8 * dg);
      }
    }
  };
#pragma unroll
  for (int b = 0; b < 4; b++) vr[b] = u32x4_t{0, 0, 0, 0};
  fetch(k0);
#pragma unroll 1
  for (int j0 = k0; j0 < kend; j0 += kAtK) {
    __syncthreads();  // every wave has read the step before
    uint32_t mk = 0, mv = 0;
#pragma unroll
    for (int i = 0; i < KI; i++) {
      const int e = tid + 256 * i;
      mag16(kr[i], mk);
      *reinterpret_cast<u32x4_t *>(ks + (e / U) * KS + 8 * (e % U)) = kr[i];
    }
#pragma unroll
    for (int b = 0; b < 4; b++) mag16(vr[b], mv);
    const bool bk = __any(nonfinite16(mk)), bv = __any(nonfinite16(mv));
    if (bv) {
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) vr[b][i] = finite_pair(vr[b][i]);
    }
    if (lane == 0) {
      bads[0][wv] = bk;
      bads[1][wv] = bv;
    }
    if (dg < U) {
      // value columns 8 dg + i of the four keys: key 16 s + 8 a + 4 f + b lies at 16 s + 8 f + 4 a + b
      const int slot = 16 * (kg >> 2) + 8 * (kg & 1) + 4 * ((kg >> 1) & 1);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t a0 = __builtin_amdgcn_perm(vr[1][i], vr[0][i], 0x05040100u);
        const uint32_t a1 = __builtin_amdgcn_perm(vr[3][i], vr[2][i], 0x05040100u);
        const uint32_t b0 = __builtin_amdgcn_perm(vr[1][i], vr[0][i], 0x07060302u);
        const uint32_t b1 = __builtin_amdgcn_perm(vr[3][i], vr[2][i], 0x07060302u);
        *reinterpret_cast<u32x2_t *>(vs + (8 * dg + 2 * i) * VS + slot) = u32x2_t{a0, a1};
        *reinterpret_cast<u32x2_t *>(vs + (8 * dg + 2 * i + 1) * VS + slot) = u32x2_t{b0, b1};
      }
    }
    __syncthreads();
    if (j0 + kAtK < kend) fetch(j0 + kAtK);
    const bool badk = (bads[0][0] | bads[0][1] | bads[0][2] | bads[0][3]) != 0;
    const bool badv = (bads[1][0] | bads[1][1] | bads[1][2] | bads[1][3]) != 0;
    if (u >= NU || j0 >= nwave) continue;  // uniform over the wave: no row of it reads these keys

    // Two chains per 32 keys, added last: the first half's high parts, and the low parts before the
    // second half's high parts, so that few roundings are at the sum's full size. Where a key
    // is not finite the second chain holds the low parts alone and is dropped from its scores.
    ff16 S[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      ff16 A, B;
#pragma unroll
      for (int i = 0; i < 16; i++) A[i] = B[i] = 0.f;
      const uint16_t *kp = ks + (32 * s + col) * KS + 8 * hf;
#pragma unroll
      for (int i = 0; i < NK; i++) {
        const fh8 a = *reinterpret_cast<const fh8 *>(kp + 16 * i);
        B = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[i], B, 0, 0, 0);
        if (i < NK / 2) A = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[i], A, 0, 0, 0);
      }
      if (badk) {
#pragma unroll
        for (int i = NK / 2; i < NK; i++)
          A = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const fh8 *>(kp + 16 * i), qh[i], A, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; i++) S[s][i] = __builtin_isfinite(A[i]) ? A[i] + B[i] : A[i];
      } else {
#pragma unroll
        for (int i = NK / 2; i < NK; i++)
          B = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const fh8 *>(kp + 16 * i), qh[i], B, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; i++) S[s][i] = A[i] + B[i];
      }
    }
    if (j0 + kAtK - 1 > limw) {  // uniform: some row does not see every key
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          if (j0 + 32 * s + 8 * (i >> 2) + 4 * hf + (i & 3) > lim) S[s][i] = -INFINITY;
    }
    float mt = S[0][0];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 16; i++) mt = fmaxf(mt, S[s][i]);
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float Mn = fmaxf(M, mt);
    if (__any(Mn > M)) {
      const float al = Mn > M ? __builtin_amdgcn_exp2f((M - Mn) * c2) : 1.f;
      L *= (double)al;
#pragma unroll
      for (int d = 0; d < ND; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) O[d][i] *= al;
      M = Mn;
    }
    const float Mu = M == -INFINITY ? 0.f : M;  // no key of this row yet: every score is -inf
    float ts[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int k = 0; k < 2; k++) {
        fh8 ph, pl;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float p = __builtin_amdgcn_exp2f((S[s][8 * k + i] - Mu) * c2);
          ts[i & 3] += p;
          const _Float16 a = (_Float16)(p * kAtUp);
          ph[i] = a;
          pl[i] = (_Float16)__builtin_fmaf(p, kAtUp, -(float)a);  // exact
        }
#pragma unroll
        for (int d = 0; d < ND; d++) {
          const fh8 a = *reinterpret_cast<const fh8 *>(vs + (32 * d + col) * VS + 32 * s + 16 * k + 8 * hf);
          O[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph, O[d], 0, 0, 0);
          O[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl, O[d], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // one half's probabilities live at a time
    }
    L += (double)((ts[0] + ts[1]) + (ts[2] + ts[3]));
    if (badv) {
      const int kn = kend - j0 < kAtK ? kend - j0 : kAtK;
#pragma unroll 1
      for (int k = 0; k < kn; k++) {
        const uint16_t *vp = Vb + (int64_t)(j0 + k) * kv_dim;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const uint16_t v = vp[32 * d + 8 * (i >> 2) + 4 * hf + (i & 3)];
            if ((v & 0x7c00u) == 0x7c00u && j0 + k <= lim) O[d][i] += (float)__builtin_bit_cast(_Float16, v);
          }
      }
    }
  }
  if (u >= NU || tb * kAtQ + col >= T) return;
  const int n = lim + 1;
  if (k0 >= n) return;  // a chunk past this row's positions has no record
  L += __shfl_xor(L, 32, 64);
  const bool whole = chunk >= n;  // the row's only chunk
  float *op = whole ? out + (int64_t)t * ldo + (int64_t)h * HD
                    : part + (((int64_t)t * (KH * G) + h) * chunks + c) * (HD + 4);
  const double f = (whole ? 1.0 / L : 1.0) * (1.0 / kAtUp);
#pragma unroll
  for (int d = 0; d < ND; d++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      ff4 o;
#pragma unroll
      for (int j = 0; j < 4; j++) o[j] = (float)((double)O[d][4 * i + j] * f);
      *reinterpret_cast<ff4 *>(op + 32 * d + 8 * i + 4 * hf) = o;
    }
  if (!whole && hf == 0) {
    op[HD] = M;
    op[HD + 1] = c2;
    *reinterpret_cast<double *>(op + HD + 2) = L;
  }
}

// Rows of more than one chunk: the chunks' sums under their largest maximum, in chunk order. One
// wave per (head, row).
template <int HD>
__global__ __launch_bounds__(256) void attention_tiles_combine_kernel(const float *__restrict__ part, int S, int heads,
                                                                      int T, int pos0, int chunk,
                                                                      float *__restrict__ out, int64_t ldo) {
  const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= (int64_t)T * heads) return;
  const int lane = threadIdx.x & 63, t = (int)(id / heads), h = (int)(id % heads);
  const int nc = (pos0 + t) / chunk + 1;
  if (nc == 1) return;
  const float *rec = part + id * S * (HD + 4);
  float m = -INFINITY;
  for (int c = 0; c < nc; c++) m = fmaxf(m, rec[c * (HD + 4) + HD]);
  double L = 0.0;
  float o[HD / 64] = {};
  for (int c = 0; c < nc; c++) {
    const float *rc = rec + c * (HD + 4);
    const float w = __builtin_amdgcn_exp2f((rc[HD] - m) * rc[HD + 1]);
    L += *reinterpret_cast<const double *>(rc + HD + 2) * (double)w;
#pragma unroll
    for (int i = 0; i < HD / 64; i++) o[i] = __builtin_fmaf(rc[lane + 64 * i], w, o[i]);
  }
  const double f = 1.0 / L;
#pragma unroll
  for (int i = 0; i < HD / 64; i++) out[(int64_t)t * ldo + (int64_t)h * HD + lane + 64 * i] = (float)((double)o[i] * f);
}

// -------------------------------------------------------------------------------------- host
// From 16 rows on: a wave's 32 columns are half used there, and it is still the faster kernel
// (fewer rows also keep the row kernels' promise that a row's bits are a single token's).
bool attention_tiles_applies(int T, int hd) { return T >= 16 && (hd == 64 || hd == 128); }

// Positions per chunk. Whole rows when the (KV head, four token blocks) workgroups alone give
// every CU two; otherwise the positions are cut so that they do, in chunks of at least 64 and
// equal to within one step.
static int tiles_chunk(int T, int heads, int kv_heads, int max_n) {
  const int G = heads / kv_heads, wgs = kv_heads * (((T + kAtQ - 1) / kAtQ * G + kAtW - 1) / kAtW);
  const int steps = (max_n + kAtK - 1) / kAtK;
  int S = (512 + wgs - 1) / wgs;
  if (wgs >= 256) S = 1;
  if (S > steps) S = steps;
  return (steps + S - 1) / S * kAtK;
}

int64_t attention_tiles_scratch_floats(int T, int heads, int kv_heads, int hd, int max_n) {
  const int chunk = tiles_chunk(T, heads, kv_heads, max_n), S = (max_n + chunk - 1) / chunk;
  return S > 1 ? (int64_t)T * heads * S * (hd + 4) : 0;
}

template <int HD>
static hipError_t tiles_launch(const float *q, int64_t ldq, int T, const uint16_t *K, const uint16_t *V, int kv_dim,
                               int heads, int kv_heads, int pos0, float scale, float *part, float *out, int64_t ldo,
                               hipStream_t st) {
  const int max_n = pos0 + T, chunk = tiles_chunk(T, heads, kv_heads, max_n), S = (max_n + chunk - 1) / chunk;
  const int G = heads / kv_heads, nz = ((T + kAtQ - 1) / kAtQ * G + kAtW - 1) / kAtW;
  // one grid dimension: the others hold 65,535 workgroups, which 512 heads of one KV head pass at 16,400 rows
  hipLaunchKernelGGL(attention_tiles_kernel<HD>, dim3((unsigned)((int64_t)kv_heads * S * nz)), dim3(256), 0, st, q, ldq,
                     K, V, kv_dim, kv_heads, G, S, nz, T, pos0, scale, chunk, part, out, ldo);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || S == 1) return e;
  hipLaunchKernelGGL(attention_tiles_combine_kernel<HD>, dim3((unsigned)(((int64_t)T * heads + 3) / 4)), dim3(256), 0, st,
                     part, S, heads, T, pos0, chunk, out, ldo);
  return hipGetLastError();
}

hipError_t attention_tiles_launch(const float *q, int64_t ldq, int T, const uint16_t *K, const uint16_t *V, int kv_dim,
                                  int heads, int kv_heads, int hd, int pos0, float scale, float *part, float *out,
                                  int64_t ldo, hipStream_t st) {
  return hd == 64 ? tiles_launch<64>(q, ldq, T, K, V, kv_dim, heads, kv_heads, pos0, scale, part, out, ldo, st)
                  : tiles_launch<128>(q, ldq, T, K, V, kv_dim, heads, kv_heads, pos0, scale, part, out, ldo, st);
}

}  // namespace wl
