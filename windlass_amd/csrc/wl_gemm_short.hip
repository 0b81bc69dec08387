// wl_gemm_short.hip - prompts of 9 to 128 tokens on the bf16 matrix cores.
//
// What bounds it: the weights' bytes (an 8B layer's 132 MB are 20 us at 6.5 TB/s) and the decode
// (about 3 VALU instructions a weight, 19 us for the layer), not the products. So every weight is
// read and decoded once for all tokens, straight from memory into the registers of the lane whose
// matrix operand it is: no LDS for weights. Tokens are multiplied in tiles of 16, 5 and 7 tiles as 6
// and 8 (the last one again). The kernels of 8 tiles by 32 rows on eight waves spill 12 to 15 registers.
//
// A workgroup owns 16 R rows and splits K over its KW waves, whose sums meet in LDS at the end in
// wave order: the launch fills the device without partial planes in memory and a launch to add
// them. The split depends on the columns alone, so a matrix gives the same bits
// alone, beside others in one launch, or as gate or up.
//
// Lane (q = l / 16, rr = l % 16) of a wave holds quarter q of row rr's 256 columns, and chunk m =
// 2 g + p is v_mfma_f32_16x16x32_bf16 with the lane's values 8 p .. 8 p + 7 of its run g of 16. Which
// columns a quarter is follows the format, so that no lane loads a byte that another uses and every
// field is a few loads of 16 bytes (in order 0 the 34-byte blocks of Q8_0 took 6 loads a run, 49 us of
// 14336 x 4096 at 9 tokens):
//   order 0 (Q4_K, Q5_K, Q6_K): q = 2 hh + ih is columns 128 hh + 32 g + 16 ih + (0..15)
//   order 1 (Q8_0, IQ4_XS):     64 q + 16 g + (0..15)
// x comes in the same order (wl_frag.h), 1 KB contiguous per chunk and 16 tokens, from L2 into
// registers.
//
// The weights are the reference DecodeRow's fp32 values rounded to bf16; products and sums are fp32.
#include "wl_gemm_short.h"

#include "wl_codecs.h"
#include "wl_device.h"
#include "wl_gemv_impl.h"

#pragma clang fp contract(off)

namespace wl {

namespace {

typedef __bf16 sb8 __attribute__((ext_vector_type(8)));
typedef float sf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  b2 v;
  v.x = (__bf16)a;  // round to nearest even (v_cvt_pk_bf16_f32)
  v.y = (__bf16)b;
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float ub(uint32_t v, int c) { return (float)((v >> (8 * c)) & 0xFF); }
__device__ __forceinline__ float sb(uint32_t v, int c) { return (float)(int8_t)(v >> (8 * c)); }

// Per format: load() fetches quarter q of a 256-column block, scale() its four runs' scales, and
// frag<M> decodes chunk M.

// d1 q - m1 (src/Quants.cs:345-346) as one fma has the reference's bits: d1 = d sc and m1 = dmin m
// are exact (17 significant bits), d1 q is exact (q < 32), and the one rounding left is the fma's.
struct SKScale { float d1[4], nm1[4]; };
__device__ __forceinline__ SKScale k_scale(const uint4 &h, int q) {
  // get_scale_min_k4 (src/Quants.cs:322-330) of the half's four sub-blocks, a byte each
  const uint32_t S = q < 2 ? (h.y & 0x3F3F3F3Fu) : ((h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u));
  const uint32_t M = q < 2 ? (h.z & 0x3F3F3F3Fu) : (((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u));
  const float d = half_lo(h.x), dmin = half_hi(h.x);
  SKScale s;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    s.d1[g] = d * ub(S, g);
    s.nm1[g] = -(dmin * ub(M, g));
  }
  return s;
}
__device__ __forceinline__ uint4 k_chunk(const SKScale &s, int g, uint32_t v0, uint32_t v1) {
  const float a = s.d1[g], b = s.nm1[g];
  auto f = [&](uint32_t v, int c) { return __builtin_fmaf(a, ub(v, c), b); };
  return make_uint4(pk_bf16(f(v0, 0), f(v0, 1)), pk_bf16(f(v0, 2), f(v0, 3)), pk_bf16(f(v1, 0), f(v1, 1)),
                    pk_bf16(f(v1, 2), f(v1, 3)));
}
__device__ __forceinline__ uint32_t dw_at(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
// the word as it stands, so that each value is one v_cvt_f32_ubyteN of it
__device__ __forceinline__ uint32_t whole(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

struct SQ4K {
  static constexpr int BYTES = 144;
  struct Raw { uint4 h, q0, q1; };
  typedef SKScale Scale;
  __device__ static void load(const uint8_t *b, int q, Raw &r) {
    const uint8_t *p = b + 16 + 64 * (q >> 1) + 16 * (q & 1);
    r.h = ldw16(b);
    r.q0 = ldw16(p);
    r.q1 = ldw16(p + 32);
  }
  __device__ static Scale scale(const Raw &r, int q) { return k_scale(r.h, q); }
  __device__ static uint4 frag(const Raw &r, const Scale &s, int, int m) {
    const int g = m >> 1, p = m & 1;
    const uint4 w = g < 2 ? r.q0 : r.q1;
    const uint32_t a = whole((dw_at(w, 2 * p) >> (4 * (g & 1))) & 0x0F0F0F0Fu);
    const uint32_t b = whole((dw_at(w, 2 * p + 1) >> (4 * (g & 1))) & 0x0F0F0F0Fu);
    return k_chunk(s, g, a, b);
  }
};

struct SQ5K {
  static constexpr int BYTES = 176;
  struct Raw { uint4 h, qh, q0, q1; };
  typedef SKScale Scale;
  __device__ static void load(const uint8_t *b, int q, Raw &r) {
    const uint8_t *p = b + 48 + 64 * (q >> 1) + 16 * (q & 1);
    r.h = ldw16(b);
    r.qh = ldw16(b + 16 + 16 * (q & 1));
    r.q0 = ldw16(p);
    r.q1 = ldw16(p + 32);
  }
  __device__ static Scale scale(const Raw &r, int q) { return k_scale(r.h, q); }
  __device__ static uint4 frag(const Raw &r, const Scale &s, int q, int m) {
    const int g = m >> 1, p = m & 1;
    const uint4 w = g < 2 ? r.q0 : r.q1;
    const int sh = 4 * (q >> 1) + g;  // the sub-block's bit of qh
    uint32_t v[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
      v[i] = whole(((dw_at(w, 2 * p + i) >> (4 * (g & 1))) & 0x0F0F0F0Fu) |
                   (((dw_at(r.qh, 2 * p + i) >> sh) & 0x01010101u) << 4));
    return k_chunk(s, g, v[0], v[1]);
  }
};

// s * v of the eight signed bytes of a, b (a product rounds once: the order of its factors is free)
__device__ __forceinline__ uint4 scaled_chunk(float s, uint32_t a, uint32_t b) {
  a = whole(a);
  b = whole(b);
  return make_uint4(pk_bf16(s * sb(a, 0), s * sb(a, 1)), pk_bf16(s * sb(a, 2), s * sb(a, 3)),
                    pk_bf16(s * sb(b, 0), s * sb(b, 1)), pk_bf16(s * sb(b, 2), s * sb(b, 3)));
}

// Blocks at 2-byte alignment come as aligned dword windows (a load at 2-byte alignment is slower than
// the window's extra dword: Q6_K 14336 x 4096 at 9 tokens 33 us with them).
struct SQ6K {
  static constexpr int BYTES = 210;
  // every field offset is a multiple of 4: the fields share the block's misalignment
  struct Raw { uint32_t l0[5], l1[5], qh[5], sc[3], dw, sh; };
  struct Scale { float ds[4]; };
  __device__ static void window(gu32 *a, uint32_t (&o)[5]) {
    const u32x4a4_t v = *reinterpret_cast<gu32x4 *>(a);
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
    o[3] = v.w;
    o[4] = ldw4(a + 4);
  }
  __device__ static void load(const uint8_t *blk, int q, Raw &r) {
    const int hh = q >> 1, ih = q & 1;
    gu32 *a = align4_down(blk);
    r.sh = misalign4(blk) * 8;
    window(a + 16 * hh + 4 * ih, r.l0);
    window(a + 16 * hh + 8 + 4 * ih, r.l1);
    window(a + 32 + 8 * hh + 4 * ih, r.qh);
    ldw12(a + 48 + 2 * hh, r.sc);
    r.dw = ldw4(a + 52);
  }
  __device__ static Scale scale(const Raw &r, int q) {
    const float d = half_lo(r.dw >> r.sh);
    Scale s;
#pragma unroll
    for (int i = 0; i < 2; i++) {  // scale bytes 2g + ih of the half's 8
      const uint32_t w = __builtin_amdgcn_alignbit(r.sc[i + 1], r.sc[i], r.sh) >> (8 * (q & 1));
      s.ds[2 * i] = d * sb(w, 0);
      s.ds[2 * i + 1] = d * sb(w, 2);
    }
    return s;
  }
  __device__ static uint4 frag(const Raw &r, const Scale &s, int, int m) {
    const int g = m >> 1, p = m & 1;
    uint32_t w[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {  // src/Quants.cs:381-392
      const uint32_t *ql = (g & 1) ? r.l1 : r.l0;
      const uint32_t L = __builtin_amdgcn_alignbit(ql[2 * p + i + 1], ql[2 * p + i], r.sh);
      const uint32_t H = __builtin_amdgcn_alignbit(r.qh[2 * p + i + 1], r.qh[2 * p + i], r.sh);
      const uint32_t v = ((L >> (4 * (g >> 1))) & 0x0F0F0F0Fu) | (((H >> (2 * g)) & 0x03030303u) << 4);
      // q - 32 per byte (0 <= q < 64): bit 7 set keeps the borrow inside its byte
      w[i] = ((v | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
    }
    return scaled_chunk(s.ds[g], w[0], w[1]);
  }
};

// Quarter q is 34-byte blocks 2q and 2q + 1 of the eight, 68 contiguous bytes: d f16 | int8[32] twice.
struct SQ80 {
  static constexpr int BYTES = 272;
  struct Raw { uint32_t w[18], sh; };  // the aligned dwords around the 68 bytes
  struct Scale { float d[2]; };
  __device__ static void load(const uint8_t *blk, int q, Raw &r) {
    const uint8_t *b = blk + 68 * q;
    gu32 *a = align4_down(b);
    r.sh = misalign4(b) * 8;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const u32x4a4_t v = *reinterpret_cast<gu32x4 *>(a + 4 * i);
      r.w[4 * i] = v.x;
      r.w[4 * i + 1] = v.y;
      r.w[4 * i + 2] = v.z;
      r.w[4 * i + 3] = v.w;
    }
    r.w[16] = ldw4(a + 16);
    r.w[17] = ldw4(a + 17);
  }
  // dword i of the 68 bytes; the quants start at byte 2 (first block) and 36
  __device__ static uint32_t dw(const Raw &r, int i) { return __builtin_amdgcn_alignbit(r.w[i + 1], r.w[i], r.sh); }
  __device__ static Scale scale(const Raw &r, int) { return Scale{{half_lo(dw(r, 0)), half_hi(dw(r, 8))}}; }
  __device__ static uint4 frag(const Raw &r, const Scale &s, int, int m) {  // src/Quants.cs:257
    const int g = m >> 1, p = m & 1, i = 4 * (g & 1) + 2 * p;
    uint32_t w[2];
#pragma unroll
    for (int k = 0; k < 2; k++)
      w[k] = g < 2 ? __builtin_amdgcn_alignbit(dw(r, i + k + 1), dw(r, i + k), 16) : dw(r, 9 + i + k);
    return scaled_chunk(s.d[g >> 1], w[0], w[1]);
  }
};

// Quarter q is sub-blocks 2q and 2q + 1 of 32: runs 0 and 1 the first's low and high nibbles.
struct SIQ4XS {
  static constexpr int BYTES = 136;
  struct Raw { uint2 h, v[4]; };
  struct Scale { float dl[2]; };
  __device__ static void load(const uint8_t *b, int q, Raw &r) {  // 8-byte aligned
    r.h = ldw8(b);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint4 v = ldw16_a2(b + 8 + 32 * q + 16 * i);
      r.v[2 * i] = make_uint2(v.x, v.y);
      r.v[2 * i + 1] = make_uint2(v.z, v.w);
    }
  }
  __device__ static Scale scale(const Raw &r, int q) {
    const float d = half_lo(r.h.x);
    const uint32_t l = r.h.y >> (8 * q), h = r.h.x >> (16 + 4 * q);  // src/IQuants.cs:69-72
    Scale s;
#pragma unroll
    for (int i = 0; i < 2; i++) s.dl[i] = d * (float)((int)(((l >> (4 * i)) & 0xF) | (((h >> (2 * i)) & 3) << 4)) - 32);
    return s;
  }
  __device__ static uint4 frag(const Raw &r, const Scale &s, int, int m) {
    const int g = m >> 1, p = m & 1;
    const uint2 w = r.v[2 * (g >> 1) + p];
    return scaled_chunk(s.dl[g >> 1], iq4_signed4((w.x >> (4 * (g & 1))) & 0x0F0F0F0Fu), iq4_signed4((w.y >> (4 * (g & 1))) & 0x0F0F0F0Fu));
  }
};

struct ShortArgs {
  ShortMat m[SHORT_MAX_MATS];  // PAIR: m[0] gate, m[1] up
  int wg0[SHORT_MAX_MATS];     // a matrix's first row group
  int nmat, nblk, T, tiles;    // token tiles of 16
  const uint4 *xf;
  int add;
  float rs;
  uint16_t *hf;  // PAIR: the results' fragments, their order
  int hord;
};

// Token tiles whose waves' sums meet in LDS at a time: a result per thread.
constexpr int short_round(int kw, int r, int nt) {
  const int n = kw * 64 / (256 * r) < 1 ? 1 : kw * 64 / (256 * r);
  return n < nt ? n : nt;
}

// One row group of 16 R rows (PAIR: 16 of gate, 16 of up) by NT token tiles.
template <class C, int R, int NT, int KW, bool PAIR>
__device__ __forceinline__ void short_body(const ShortArgs &a, const ShortMat &mat, int row0, float *red) {
  constexpr int XD = NT <= 2 ? 4 : 2;  // x chunks held: XD - 1 on their way
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, rr = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b0 = (int)((int64_t)a.nblk * wv / KW), b1 = (int)((int64_t)a.nblk * (wv + 1) / KW);
  const uint8_t *wr[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    if constexpr (PAIR) wr[r] = a.m[r].w + (int64_t)(row0 + rr) * mat.row_bytes;  // rows are whole groups
    else wr[r] = mat.w + (int64_t)min(row0 + 16 * r + rr, mat.rows - 1) * mat.row_bytes;
  }
  const uint4 *xs[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) xs[t] = a.xf + (int64_t)min(t, a.tiles - 1) * a.nblk * 512 + lane;
  sf4 acc[R][NT];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[r][t] = sf4{0.f, 0.f, 0.f, 0.f};
  if (b0 < b1) {
    typename C::Raw nxt[R];
    uint4 x[XD][NT];
    auto fetch_x = [&](int c, uint4 (&o)[NT]) {  // chunk c of the row's 8 nblk; past the wave's: its last
      const int64_t at = (int64_t)min(c, 8 * b1 - 1) * 64;
#pragma unroll
      for (int t = 0; t < NT; t++) o[t] = xs[t][at];
    };
#pragma unroll
    for (int r = 0; r < R; r++) C::load(wr[r] + (int64_t)b0 * C::BYTES, q, nxt[r]);
#pragma unroll
    for (int c = 0; c < XD - 1; c++) fetch_x(8 * b0 + c, x[c]);
#pragma unroll 1
    for (int b = b0; b < b1; b++) {
      typename C::Raw cur[R];
      typename C::Scale sc[R];
      const int bn = b + 1 < b1 ? b + 1 : b;  // past the end: the last again (unused)
#pragma unroll
      for (int r = 0; r < R; r++) {
        cur[r] = nxt[r];
        C::load(wr[r] + (int64_t)bn * C::BYTES, q, nxt[r]);
      }
#pragma unroll
      for (int r = 0; r < R; r++) sc[r] = C::scale(cur[r], q);
#pragma unroll
      for (int m = 0; m < 8; m++) {
        fetch_x(8 * b + m + XD - 1, x[(m + XD - 1) % XD]);
#pragma unroll
        for (int r = 0; r < R; r++) {
          const sb8 w = __builtin_bit_cast(sb8, C::frag(cur[r], sc[r], q, m));
#pragma unroll
          for (int t = 0; t < NT; t++)
            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(sb8, x[m % XD][t]), acc[r][t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // a chunk's decode stays with its products
      }
    }
  }
  // the waves' sums in wave order, TR token tiles at a time: lane holds rows 4 q .. 4 q + 3 of
  // token rr of a tile
  constexpr int TR = short_round(KW, R, NT);
  sf4 *red4 = reinterpret_cast<sf4 *>(red);
#pragma unroll
  for (int t1 = 0; t1 < NT; t1 += TR) {
    if (t1) __syncthreads();  // the round before is read
#pragma unroll
    for (int t = 0; t < TR; t++)
      if (t1 + t < NT) {
#pragma unroll
        for (int r = 0; r < R; r++) red4[((wv * TR + t) * R + r) * 64 + rr * 4 + q] = acc[r][t1 + t < NT ? t1 + t : 0];
      }
    __syncthreads();
    if constexpr (PAIR) {
      for (int el = tid; el < TR * 256; el += KW * 64) {
        const int t = el >> 8, e = el & 255, tok = 16 * (t1 + t) + (e >> 4);
        float g = 0.f, u = 0.f;
#pragma unroll
        for (int w = 0; w < KW; w++) {
          g += red[((w * TR + t) * 2) * 256 + e];
          u += red[((w * TR + t) * 2 + 1) * 256 + e];
        }
        if (t1 + t < NT && tok < a.tiles * 16) {  // tokens past T in the last tile: any value, never stored in y
          const int row = row0 + (e & 15);
          const __bf16 h = (__bf16)silu_mul(g, u);
          a.hf[frag_at(tok, row & ~7, mat.rows, a.hord) * 8 + (row & 7)] = __builtin_bit_cast(uint16_t, h);
        }
      }
    } else {
      for (int el = tid; el < TR * R * 256; el += KW * 64) {
        const int t = el / (256 * R), r = (el >> 8) % R, e = el & 255, tok = 16 * (t1 + t) + (e >> 4);
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < KW; w++) s += red[((w * TR + t) * R + r) * 256 + e];
        const int row = row0 + 16 * r + (e & 15);
        if (t1 + t < NT && tok < a.T && row < mat.rows) {
          float *yp = mat.y + (int64_t)tok * mat.ldy + row;
          *yp = a.add ? add_scaled(*yp, s, a.rs) : s;
        }
      }
    }
  }
}

template <int R, int NT, int KW, bool PAIR>
__global__ __launch_bounds__(64 * KW) void short_kernel(ShortArgs a) {
  __shared__ float red[KW * short_round(KW, R, NT) * R * 256];
  const int rg = blockIdx.x;
  int k = 0;
  if constexpr (!PAIR) {
    if (a.nmat > 1 && rg >= a.wg0[1]) k = 1;
    if (a.nmat > 2 && rg >= a.wg0[2]) k = 2;
  }
  const ShortMat &m = a.m[k];
  const int row0 = (rg - a.wg0[k]) * (PAIR ? 16 : 16 * R);
  switch (m.type) {
    case 8: short_body<SQ80, R, NT, KW, PAIR>(a, m, row0, red); break;
    case 12: short_body<SQ4K, R, NT, KW, PAIR>(a, m, row0, red); break;
    case 13: short_body<SQ5K, R, NT, KW, PAIR>(a, m, row0, red); break;
    case 14: short_body<SQ6K, R, NT, KW, PAIR>(a, m, row0, red); break;
    case 23: short_body<SIQ4XS, R, NT, KW, PAIR>(a, m, row0, red); break;
  }
}

// ------------------------------------------------------------------------------- operands
// A thread per 16-byte piece; tokens past T in the last tile repeat token T - 1 here. Pieces that a norm
// or gate and up write leave those places as they are or hold any value: an MFMA's columns are
// independent, and the results of tokens past T are never stored.
__global__ __launch_bounds__(256) void short_frag_kernel(const float *__restrict__ x, int T, int cols, int64_t n,
                                                         int ord, uint4 *__restrict__ xf) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int nblk = cols >> 8, lane = (int)(i & 63), m = (int)(i >> 6) & 7;
  const int b = (int)((i >> 9) % nblk), tt = (int)((i >> 9) / nblk);
  const int q = lane >> 4, t = min(16 * tt + (lane & 15), T - 1);
  const int k = 256 * b + (ord ? 64 * q + 8 * m : 128 * (q >> 1) + 32 * (m >> 1) + 16 * (q & 1) + 8 * (m & 1));
  float v[8];
  ld_x8(x + (int64_t)t * cols + k, v);
  xf[i] = make_uint4(pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]), pk_bf16(v[4], v[5]), pk_bf16(v[6], v[7]));
}

template <int R, int NT, int KW, bool PAIR>
hipError_t go(const ShortArgs &a, int groups, hipStream_t st) {
  hipLaunchKernelGGL((short_kernel<R, NT, KW, PAIR>), dim3((unsigned)groups), dim3(64 * KW), 0, st, a);
  return hipGetLastError();
}

constexpr int kShortT = 128;  // tokens at most: 8 tiles' accumulators

template <int R, int KW, bool PAIR>
hipError_t dispatch_kw(const ShortArgs &a, int groups, hipStream_t st) {
  switch (a.tiles) {
    case 1: return go<R, 1, KW, PAIR>(a, groups, st);
    case 2: return go<R, 2, KW, PAIR>(a, groups, st);
    case 3: return go<R, 3, KW, PAIR>(a, groups, st);
    case 4: return go<R, 4, KW, PAIR>(a, groups, st);
    case 5:
    case 6: return go<R, 6, KW, PAIR>(a, groups, st);
    default: return go<R, 8, KW, PAIR>(a, groups, st);
  }
}

// Waves that share a row's columns: four, whose longer walks pay the first and last memory round trip
// once for more blocks, or eight for rows past 10,240 columns, which are most of the time of matrices
// of few rows (45 tokens: Q4_K 14336 x 4096 25.4 us with four and 28.7 with eight, 28672 x 8192 76.6 and
// 85.1, 4096 x 4096 12.1 and 11.5, 4096 x 14336 31.5 and 30.2; at 9 tokens 22.4 and 19.7). By the columns
// alone, so that a matrix has the same bits in every launch.
template <int R, bool PAIR>
hipError_t dispatch(const ShortArgs &a, int groups, hipStream_t st) {
  return a.nblk > 40 ? dispatch_kw<R, 8, PAIR>(a, groups, st) : dispatch_kw<R, 4, PAIR>(a, groups, st);
}

ShortArgs args_of(int cols, const void *xf, int T) {
  ShortArgs a{};
  a.nblk = cols / 256;
  a.T = T;
  a.tiles = (T + 15) / 16;
  a.xf = (const uint4 *)xf;
  return a;
}

}  // namespace

bool short_type(int type) { return type == 8 || type == 12 || type == 13 || type == 14 || type == 23; }

bool short_applies(int type, int T, int64_t cols) { return short_type(type) && T > 8 && T <= kShortT && cols % 256 == 0; }

hipError_t short_frag_launch(const float *x, int T, int cols, int ord, void *xf, hipStream_t st) {
  const int64_t n = frag_bytes(T, cols, ord) / 16;
  hipLaunchKernelGGL(short_frag_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, T, cols, n, ord,
                     (uint4 *)xf);
  return hipGetLastError();
}

hipError_t short_matmul_launch(const ShortMat *mats, int n, int cols, const void *xf, int T, bool add, float rs,
                               int num_cu, hipStream_t st) {
  if (n < 1 || n > SHORT_MAX_MATS || cols <= 0 || cols % 256 || T < 1 || T > kShortT || !xf) return hipErrorInvalidValue;
  ShortArgs a = args_of(cols, xf, T);
  a.nmat = n;
  a.add = add;
  a.rs = rs;
  int64_t rows = 0;
  for (int i = 0; i < n; i++) {
    if (!short_type(mats[i].type) || short_order(mats[i].type) != short_order(mats[0].type) || mats[i].rows < 1)
      return hipErrorInvalidValue;
    a.m[i] = mats[i];
    rows += mats[i].rows;
  }
  // 32 rows a workgroup read x half as often; 16 where those would leave CUs without a workgroup
  // (Q4_K, 45 tokens, eight waves: 14336 x 4096 32.7 us with 16 rows and 28.6 with 32; 4096 x 4096 11.8
  // and 14.4)
  const int R = rows / 32 >= num_cu ? 2 : 1;
  int groups = 0;
  for (int i = 0; i < n; i++) {
    a.wg0[i] = groups;
    groups += (mats[i].rows + 16 * R - 1) / (16 * R);
  }
  return R == 2 ? dispatch<2, false>(a, groups, st) : dispatch<1, false>(a, groups, st);
}

hipError_t short_swiglu_launch(const ShortMat &gate, const ShortMat &up, int cols, const void *xf, int T, void *hf,
                               int hord, hipStream_t st) {
  if (cols <= 0 || cols % 256 || T < 1 || T > kShortT || !xf || !hf || !short_type(gate.type) || gate.type != up.type ||
      gate.rows != up.rows || gate.rows % 256 || gate.row_bytes != up.row_bytes)
    return hipErrorInvalidValue;
  ShortArgs a = args_of(cols, xf, T);
  a.nmat = 1;
  a.m[0] = gate;
  a.m[1] = up;
  a.hf = (uint16_t *)hf;
  a.hord = hord;
  return dispatch<2, true>(a, gate.rows / 16, st);
}

}  // namespace wl
