// wl_moe_mma.hip - routed experts of a prompt (more than 8 tokens) on the matrix cores: Q4_K and
// Q6_K experts, each expert's weights read once for all of its tokens (MoeFfn,
// src/Transformer.cs:253-311).
//
// What bounds it: at 128 experts of 2048 x 768, top-8 and 300 tokens every expert is chosen, so
// the 378 MB of weights (about 60 us at 6.3 TB/s) are the floor; the products are 45 GFLOP on the
// matrix cores in two fp16 parts. The passes of 8 tokens it replaces read the chosen experts
// again in every pass of 8 (38 passes, 3,648 us).
//
// Arithmetic, at fp32's precision: a weight is an exact fp16 integer (wl_fmma_codec.h), a
// token's 256 activations of a super-block are scaled by a power of two and split into
// hi = fp16(x f), lo = fp16(x f - hi), 22 significant bits down to 2^-17 of the 256's largest value
// (2^-39 of it below), and the exact products accumulate into fp32, the parts apart (the lo sums round
// 2^11 times finer). Q4_K's quants enter as n - 8, with the sub-block's 8 d sc - dmin m as the factor of
// its sum of x (a 16x16x4 fp32 MFMA): the two large terms that nearly cancel in n sc and the minimum
// never become sums of their own (error against 64 bits at 300 tokens of 128 experts 5.2e-7 with n, 2.4e-7
// so, 3.7e-7 row by row in fp32; over 24 drawn shapes, some with columns 30 to 10,000 times the others,
// 2.2e-7 to 2.8e-7 against 2.9e-7 to 4.2e-7 row by row). A super-block's sum is then scaled by d and 1/f
// and added in order, so a token's result depends neither on the other tokens nor on its place in a
// tile.
//
// Launches: route (one wave per token), plan (one workgroup per expert numbers its pairs), the
// tokens' parts, gate/up with the SiLU, the hidden rows' parts, down, combine.
#include "wl_fmma_codec.h"
#include "wl_gemv_impl.h"
#include "wl_moe.h"

#pragma clang fp contract(off)

namespace wl {

// ------------------------------------------------------------------------------------- plan
// Pairs (token, choice) numbered experts ascending, tokens ascending within an expert, and cut
// into tiles of at most TT pairs of one expert. Block e counts every expert's pairs in LDS, so no
// block waits for another, and numbers expert e's pairs in order with ballots.
__global__ __launch_bounds__(256) void moe_many_plan_kernel(const int *__restrict__ sel, const float *__restrict__ wts,
                                                            int P, int k, int n, int TT, MoeMany m) {
  extern __shared__ int moe_hist[];
  __shared__ int red[2][4], wtot[4];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int i = tid; i < n; i += 256) moe_hist[i] = 0;
  __syncthreads();
  for (int i = tid; i < P; i += 256) atomicAdd(&moe_hist[sel[i]], 1);
  __syncthreads();
  int base = 0, tbase = 0;
  for (int i = tid; i < e; i += 256) {
    base += moe_hist[i];
    tbase += (moe_hist[i] + TT - 1) / TT;
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    base += __shfl_xor(base, o, 64);
    tbase += __shfl_xor(tbase, o, 64);
  }
  if (lane == 0) {
    red[0][wv] = base;
    red[1][wv] = tbase;
  }
  __syncthreads();
  base = red[0][0] + red[0][1] + red[0][2] + red[0][3];
  tbase = red[1][0] + red[1][1] + red[1][2] + red[1][3];
  const int cnt = moe_hist[e], nt = (cnt + TT - 1) / TT;
  if (e == n - 1 && tid == 0) *m.ntiles = tbase + nt;
  for (int i = tid; i < nt; i += 256)
    m.tiles[tbase + i] = MoeTile{e, base + i * TT, cnt - i * TT < TT ? cnt - i * TT : TT};
  if (cnt == 0) return;  // uniform
  int at = base;
  for (int i0 = 0; i0 < P; i0 += 256) {
    const int i = i0 + tid;
    const bool mine = i < P && sel[i] == e;
    const uint64_t b = __ballot(mine);
    if (lane == 0) wtot[wv] = __popcll(b);
    __syncthreads();
    int before = at;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      before += w < wv ? wtot[w] : 0;
      at += wtot[w];
    }
    if (mine) {
      const int pos = before + __popcll(b & ((1ull << lane) - 1)), t = i / k;
      int r = 0;  // this choice's place among the token's, experts ascending (the combine's order)
      for (int j = 0; j < k; j++) r += sel[t * k + j] < e ? 1 : 0;
      m.pair_tok[pos] = t;
      m.comb_pair[t * k + r] = pos;
      m.comb_w[t * k + r] = wts[i];
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------ parts
// x [rows][cols] fp32 -> per (row, super-block): 64 operand chunks of 16 bytes, chunk
// (2 m + part) * 4 + q holding the part's values (q, m); the sub-blocks' sums of x f [8]
// (sub-block 2q + h at 4h + q) and 1/f. One wave per (row, super-block).
template <class C>
__global__ __launch_bounds__(256) void moe_parts_kernel(const float *__restrict__ x, int64_t rows, int nsb,
                                                        uint4 *__restrict__ parts, float *__restrict__ sums,
                                                        float *__restrict__ inv) {
  const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= rows * nsb) return;
  const int lane = threadIdx.x & 63, part = lane >> 5, m = (lane & 31) >> 2, q = lane & 3;
  const float *xs = x + id * 256;
  const float4 a = *reinterpret_cast<const float4 *>(xs + C::xoff4(q, m, 0));
  const float4 b = *reinterpret_cast<const float4 *>(xs + C::xoff4(q, m, 1));
  float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float t = fabsf(v[i]);
    mx = t < INFINITY ? fmaxf(mx, t) : mx;  // NaN and infinities take no part
  }
  mx = wave_max_f(mx);
  float f, iv;
  unit_scale(mx, f, iv);
  fh8 o;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    // the chunk's order of each four values (WQ4K: 0, 2, 1, 3)
    const int j = C::SWAP && (i & 3) == 1 ? i + 1 : C::SWAP && (i & 3) == 2 ? i - 1 : i;
    const float X = v[j] * f;
    const _Float16 hi = (_Float16)X;
    o[i] = part == 0 ? hi : (_Float16)(__builtin_isinf(X) ? 0.f : X - (float)hi);  // an infinity is all hi
  }
  parts[id * 64 + (2 * m + part) * 4 + q] = __builtin_bit_cast(uint4, o);
  if constexpr (C::MINS) {
    float s[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      s[h] = ((v[4 * h] + v[4 * h + 1]) + (v[4 * h + 2] + v[4 * h + 3])) * f;
      s[h] += __shfl_xor(s[h], 4, 64);
      s[h] += __shfl_xor(s[h], 8, 64);
      s[h] += __shfl_xor(s[h], 16, 64);
    }
    if (lane < 4) {
      sums[id * 8 + q] = s[0];
      sums[id * 8 + 4 + q] = s[1];
    }
  }
  if (lane == 0) inv[id] = iv;
}

// --------------------------------------------------------------------------------- products
// A workgroup of four waves owns one tile of pairs (up to 16 NT of one expert) and 128 row
// slots of its weights: for PAIR each wave has 16 rows of gate and the same of up, otherwise 32
// rows of one matrix. Per super-block the pairs' parts (NT * 16 KB) pass through LDS, read by the
// four waves, while the next super-block's parts and weights are on their way in registers; the
// weights go from memory to their lane. One LDS buffer, so that several workgroups share a CU.
// Workgroups of one tile run on one XCD: they share the pairs' parts in its L2.
struct MoeGemm {
  MoeMany m;
  const uint8_t *w, *w2;
  int64_t row_bytes, expert_bytes;
  int rows, nsb;
  const u32x4_t *parts;
  const float *sums, *inv;
  int by_pair;  // parts by pair (down) or by token (gate/up)
  float *y;     // [pair][rows]
};

template <class C, bool PAIR, int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void moe_many_kernel(MoeGemm a) {
  __shared__ u32x4_t xs[NT * 64 * 16];
  __shared__ float xsum[NT * 8 * 16], xinv[NT * 16];
  const int rt = a.rows / (PAIR ? 64 : 128);
  const int xcd = blockIdx.x & 7, j0 = blockIdx.x >> 3;
  const int tile = xcd + 8 * (j0 / rt), r0 = (j0 % rt) * (PAIR ? 64 : 128);
  if (tile >= *a.m.ntiles) return;  // uniform
  const MoeTile T = a.m.tiles[tile];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q = lane >> 4, rr = lane & 15;
  // this thread's staging: slot rr of each 16, chunks q + 4 wv + 16 i
  int64_t src[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int s = 16 * t + rr, p = T.first + (s < T.n ? s : T.n - 1);  // past the tile: its last pair again
    src[t] = (int64_t)(a.by_pair ? p : a.m.pair_tok[p]) * a.nsb;
  }
  const int ss = tid & (16 * NT - 1), sg = tid / (16 * NT);  // sums: slot and first sub-block
  const int64_t ssrc = (int64_t)(a.by_pair ? T.first + min(ss, T.n - 1) : a.m.pair_tok[T.first + min(ss, T.n - 1)]) * a.nsb;
  const uint8_t *wr[2];
  const uint8_t *we = a.w + T.expert * a.expert_bytes;
  if constexpr (PAIR) {
    const int64_t ro = (int64_t)(r0 + 16 * wv + rr) * a.row_bytes;
    wr[0] = we + ro;
    wr[1] = a.w2 + T.expert * a.expert_bytes + ro;
  } else {
    wr[0] = we + (int64_t)(r0 + 32 * wv + rr) * a.row_bytes;
    wr[1] = wr[0] + 16 * a.row_bytes;
  }
  typename C::Raw raw[2];
  u32x4_t st[NT][4];
  float ssv[NT] = {}, siv = 0.f;
  auto fetch = [&](int b) {
    C::load(wr[0] + (int64_t)b * C::BYTES, q, raw[0]);
    C::load(wr[1] + (int64_t)b * C::BYTES, q, raw[1]);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) st[t][i] = a.parts[(src[t] + b) * 64 + q + 4 * wv + 16 * i];
    if constexpr (C::MINS) {
      // 8 sums of 16 NT slots over 256 threads: NT/2 each (NT = 1: half of the threads)
#pragma unroll
      for (int i = 0; i < (NT + 1) / 2; i++) {
        const int g = sg + i * (16 / NT);
        ssv[i] = g < 8 ? a.sums[(ssrc + b) * 8 + g] : 0.f;
      }
    }
    if (tid < 16 * NT) siv = a.inv[ssrc + b];
  };
  ff4 acc[2][NT];
#pragma unroll
  for (int w = 0; w < 2; w++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[w][t] = ff4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
#pragma unroll 1
  for (int b = 0; b < a.nsb; b++) {
    __syncthreads();  // every wave has read the super-block before
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) xs[(t * 64 + q + 4 * wv + 16 * i) * 16 + rr] = st[t][i];
    if constexpr (C::MINS) {
#pragma unroll
      for (int i = 0; i < (NT + 1) / 2; i++) {
        const int g = sg + i * (16 / NT);
        if (g < 8) xsum[(g * NT + (ss >> 4)) * 16 + (ss & 15)] = ssv[i];
      }
    }
    if (tid < 16 * NT) xinv[tid] = siv;
    typename C::Raw cur[2] = {raw[0], raw[1]};
    __syncthreads();
    fetch(b + 1 < a.nsb ? b + 1 : b);  // past the end: the last again (valid, unused)
    // both weights share the reads of the parts, or (wide accumulators) one after the other
    constexpr int G = C::NF * NT > 4 ? 1 : 2;
#pragma unroll
    for (int w0 = 0; w0 < 2; w0 += G) {
      typename C::Scale sc[G];
      ff4 acc1[G][NT][C::NF], acc2[G][NT][C::NF];  // the sums of the hi and of the lo parts
#pragma unroll
      for (int w = 0; w < G; w++) {
        sc[w] = C::scale(cur[w0 + w], q);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
          for (int n = 0; n < C::NF; n++) acc1[w][t][n] = acc2[w][t][n] = ff4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int mm = 0; mm < 8; mm++) {
        fh8 f[G][C::NF];
#pragma unroll
        for (int w = 0; w < G; w++) C::frag(cur[w0 + w], sc[w], q, mm, f[w]);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const fh8 hi = __builtin_bit_cast(fh8, xs[(t * 64 + mm * 8 + q) * 16 + rr]);
          const fh8 lo = __builtin_bit_cast(fh8, xs[(t * 64 + mm * 8 + 4 + q) * 16 + rr]);
#pragma unroll
          for (int w = 0; w < G; w++)
#pragma unroll
            for (int n = 0; n < C::NF; n++) {
              acc1[w][t][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, f[w][n], acc1[w][t][n], 0, 0, 0);
              acc2[w][t][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, f[w][n], acc2[w][t][n], 0, 0, 0);
            }
        }
        if ((mm & 1) || G == 1) __builtin_amdgcn_sched_barrier(0);  // one or two chunks' operands live at a time
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const ff4 iv = *reinterpret_cast<const ff4 *>(&xinv[16 * t + 4 * q]);
#pragma unroll
        for (int w = 0; w < G; w++) {
          const float d = C::d(cur[w0 + w]);
          ff4 &o = acc[w0 + w][t];
          if constexpr (C::MINS) {
            ff4 Mn = {0.f, 0.f, 0.f, 0.f};
            Mn = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum[(q * NT + t) * 16 + rr], sc[w].mlo, Mn, 0, 0, 0);
            Mn = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum[((4 + q) * NT + t) * 16 + rr], sc[w].mhi, Mn, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++)
              o[i] = __builtin_fmaf(__builtin_fmaf(d, acc1[w][t][0][i] + acc2[w][t][0][i], Mn[i]), iv[i], o[i]);
          } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
              o[i] = __builtin_fmaf(d * __builtin_fmaf(16.f, acc1[w][t][1][i] + acc2[w][t][1][i],
                                                       acc1[w][t][0][i] + acc2[w][t][0][i]),
                                    iv[i], o[i]);
          }
        }
      }
    }
  }
  // lane: row rr of its 16-row tile, pairs 16 t + 4 q + i
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int s = 16 * t + 4 * q + i;
      if (s < T.n) {
        float *yp = a.y + (int64_t)(T.first + s) * a.rows + r0;
        if constexpr (PAIR) {
          yp[16 * wv + rr] = silu_mul(acc[0][t][i], acc[1][t][i]);
        } else {
          yp[32 * wv + rr] = acc[0][t][i];
          yp[32 * wv + 16 + rr] = acc[1][t][i];
        }
      }
    }
}

// out[t] = the token's pairs added in ascending expert order, w * y each (:289-293).
__global__ __launch_bounds__(256) void moe_many_combine_kernel(MoeMany m, const float *__restrict__ y, int T, int k,
                                                               int embd, float *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int e4 = embd / 4;
  if (i >= (int64_t)T * e4) return;
  const int t = (int)(i / e4), d = (int)(i % e4);
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int j = 0; j < k; j++) {
    const float w = m.comb_w[t * k + j];
    const float4 v = reinterpret_cast<const float4 *>(y + (int64_t)m.comb_pair[t * k + j] * embd)[d];
    o.x += w * v.x;
    o.y += w * v.y;
    o.z += w * v.z;
    o.w += w * v.w;
  }
  reinterpret_cast<float4 *>(out + (int64_t)t * embd)[d] = o;
}

// ------------------------------------------------------------------------------------- host
static bool many_type(int t) { return t == 12 || t == 14; }

// More than one pass of 8 tokens, K-quant experts whose rows are whole 256-blocks, float
// products; experts the plan's counters hold in 32 KB of LDS.
bool moe_many_applies(int gu_type, int d_type, int T, int ne, int ff, int embd) {
  return T > MOE_MAX_T && many_type(gu_type) && many_type(d_type) && ne <= 8192 && ff % 256 == 0 && embd % 256 == 0;
}

// Token tiles of 16 NT pairs: the expected pairs per expert and some (their spread), so that
// most experts are one tile and their weights are read once.
static int many_nt(int T, int k, int ne) {
  const int avg = T * k / ne;
  return avg <= 8 ? 1 : avg <= 24 ? 2 : 4;
}

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }

static int many_max_tiles(int T, int k, int ne) {
  const int P = T * k, TT = 16 * many_nt(T, k, ne);
  return (P < ne ? P : ne) + P / TT;
}

// Scratch: sel | wts | prob | the plan | parts, sums and scales of x, then of h | h | y.
struct ManyLayout {
  size_t sel, wts, prob, ntiles, tiles, tok, comb, cw, xp, xsum, xinv, hp, hsum, hinv, h, y, total;
};
static ManyLayout many_layout(int T, int k, int ne, int ff, int embd) {
  ManyLayout s{};
  const size_t P = (size_t)T * k;
  size_t o = 0;
  auto take = [&](size_t &f, size_t bytes) { f = o; o = al256(o + bytes); };
  take(s.sel, P * 4);
  take(s.wts, P * 4);
  take(s.prob, (size_t)T * ne * 4);
  take(s.ntiles, 4);
  take(s.tiles, sizeof(MoeTile) * many_max_tiles(T, k, ne));
  take(s.tok, P * 4);
  take(s.comb, P * 4);
  take(s.cw, P * 4);
  take(s.xp, (size_t)T * embd * 4);
  take(s.xsum, (size_t)T * embd / 32 * 4);
  take(s.xinv, (size_t)T * embd / 256 * 4);
  take(s.hp, P * ff * 4);
  take(s.hsum, P * ff / 32 * 4);
  take(s.hinv, P * ff / 256 * 4);
  take(s.h, P * ff * 4);
  take(s.y, P * embd * 4);
  s.total = o;
  return s;
}

int64_t moe_many_scratch_bytes(int T, int k, int ne, int ff, int embd) {
  return (int64_t)many_layout(T, k, ne, ff, embd).total;
}

static hipError_t parts_launch(int type, const float *x, int64_t rows, int cols, uint8_t *p, uint8_t *sums, uint8_t *inv,
                               hipStream_t st) {
  const int nsb = cols / 256;
  const dim3 grid((unsigned)((rows * nsb + 3) / 4));
  if (type == 12)
    hipLaunchKernelGGL(moe_parts_kernel<WQ4K>, grid, dim3(256), 0, st, x, rows, nsb, (uint4 *)p, (float *)sums, (float *)inv);
  else
    hipLaunchKernelGGL(moe_parts_kernel<WQ6K>, grid, dim3(256), 0, st, x, rows, nsb, (uint4 *)p, (float *)sums, (float *)inv);
  return hipGetLastError();
}

template <class C, bool PAIR>
static hipError_t many_gemm(const MoeGemm &a, int nt, int max_tiles, hipStream_t st) {
  const int rt = a.rows / (PAIR ? 64 : 128);
  const dim3 grid((unsigned)((max_tiles + 7) / 8 * 8 * rt));
  switch (nt) {
    case 1: hipLaunchKernelGGL((moe_many_kernel<C, PAIR, 1>), grid, dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((moe_many_kernel<C, PAIR, 2>), grid, dim3(256), 0, st, a); break;
    default: hipLaunchKernelGGL((moe_many_kernel<C, PAIR, 4>), grid, dim3(256), 0, st, a); break;
  }
  return hipGetLastError();
}

hipError_t moe_many_launch(const MoeLaunch &l, void *scratch, hipStream_t st) {
  if (!moe_many_applies(l.gu_type, l.d_type, MOE_MAX_T + 1, l.ne, l.ff, l.embd) || l.T < 1 || l.T > MOE_MANY_T ||
      l.gu_int || l.d_int || !scratch || l.k < 1 || l.k > MOE_MAX_K || l.k > l.ne)
    return hipErrorInvalidValue;
  const ManyLayout s = many_layout(l.T, l.k, l.ne, l.ff, l.embd);
  uint8_t *b = (uint8_t *)scratch;
  const int P = l.T * l.k, nt = many_nt(l.T, l.k, l.ne), max_tiles = many_max_tiles(l.T, l.k, l.ne);
  int *sel = (int *)(b + s.sel);
  float *wts = (float *)(b + s.wts);
  MoeMany m{};
  m.ntiles = (int *)(b + s.ntiles);
  m.tiles = (MoeTile *)(b + s.tiles);
  m.pair_tok = (int *)(b + s.tok);
  m.comb_pair = (int *)(b + s.comb);
  m.comb_w = (float *)(b + s.cw);
  hipError_t e = route_launch(l.logits, l.T, l.ne, l.k, l.renorm, sel, wts, (float *)(b + s.prob), st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(moe_many_plan_kernel, dim3(l.ne), dim3(256), (size_t)l.ne * 4, st, sel, wts, P, l.k, l.ne, 16 * nt, m);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = parts_launch(l.gu_type, l.x, l.T, l.embd, b + s.xp, b + s.xsum, b + s.xinv, st)) != hipSuccess) return e;
  MoeGemm g{};
  g.m = m;
  g.w = l.gate;
  g.w2 = l.up;
  g.row_bytes = l.gu_row_bytes;
  g.expert_bytes = (int64_t)l.ff * l.gu_row_bytes;
  g.rows = l.ff;
  g.nsb = l.embd / 256;
  g.parts = (const u32x4_t *)(b + s.xp);
  g.sums = (const float *)(b + s.xsum);
  g.inv = (const float *)(b + s.xinv);
  g.by_pair = 0;
  g.y = (float *)(b + s.h);
  e = l.gu_type == 12 ? many_gemm<WQ4K, true>(g, nt, max_tiles, st) : many_gemm<WQ6K, true>(g, nt, max_tiles, st);
  if (e != hipSuccess) return e;
  if ((e = parts_launch(l.d_type, g.y, P, l.ff, b + s.hp, b + s.hsum, b + s.hinv, st)) != hipSuccess) return e;
  MoeGemm d = g;
  d.w = l.down;
  d.w2 = nullptr;
  d.row_bytes = l.d_row_bytes;
  d.expert_bytes = (int64_t)l.embd * l.d_row_bytes;
  d.rows = l.embd;
  d.nsb = l.ff / 256;
  d.parts = (const u32x4_t *)(b + s.hp);
  d.sums = (const float *)(b + s.hsum);
  d.inv = (const float *)(b + s.hinv);
  d.by_pair = 1;
  d.y = (float *)(b + s.y);
  e = l.d_type == 12 ? many_gemm<WQ4K, false>(d, nt, max_tiles, st) : many_gemm<WQ6K, false>(d, nt, max_tiles, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(moe_many_combine_kernel, dim3((unsigned)(((int64_t)l.T * l.embd / 4 + 255) / 256)), dim3(256), 0, st,
                     m, d.y, l.T, l.k, l.embd, l.out);
  return hipGetLastError();
}

}  // namespace wl
