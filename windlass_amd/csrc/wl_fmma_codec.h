// wl_fmma_codec.h - Q4_K and Q6_K weights as exact fp16 integers for v_mfma_f32_16x16x32_f16, and
// the power-of-two scaling of the fp32 activations that meet them as two fp16 parts.
//
// Lane (q = l / 16, rr = l % 16) of a wave holds quarter q of row rr's super-block (64 values) and
// gives MFMA m = 0..7 its eight values of operand column rr, k = 8q .. 8q + 7. xoff(q, m, i) is
// the place within the super-block of the i-th of those eight values: the activations' operand
// chunks are laid out in the same order.
#pragma once
#include "wl_device.h"

namespace wl {

typedef _Float16 fh2 __attribute__((ext_vector_type(2)));
typedef _Float16 fh4 __attribute__((ext_vector_type(4)));
typedef _Float16 fh8 __attribute__((ext_vector_type(8)));
typedef float ff4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ fh2 as_fh2(uint32_t u) { return __builtin_bit_cast(fh2, u); }

// A unit's scale: f = 2^(15 - e) for the largest finite |x| = m 2^e (m in [0.5, 1)), and 1/f;
// both powers of two, clamped to the normal range. An all-zero (or non-finite) unit takes f = 1.
__device__ __forceinline__ void unit_scale(float mx, float &f, float &inv) {
  if (!(mx > 0.f)) {
    f = 1.f;
    inv = 1.f;
    return;
  }
  int e;
  frexpf(mx, &e);
  int s = 15 - e;
  s = s > 126 ? 126 : s;
  f = ldexpf(1.f, s);
  inv = ldexpf(1.f, -s);
}

// ------------------------------------------------------------------------------------ Q4_K
// Quarter q of a super-block is sub-block pair q: qs bytes 32q..32q+31, whose low nibbles are
// values 64q + i and high nibbles 64q + 32 + i (src/Quants.cs:333-351). MFMA m takes the lane's
// qs dword m (bytes 4m..4m+3 of the pair) as the values 64q + {4m, 4m+2, 4m+1, 4m+3} and
// 64q + 32 + {4m, 4m+2, 4m+1, 4m+3}. The quants enter centred: each fp16 pair is (dword & mask) |
// 0x6400 (1024 + n, or 1024 + 16 n), less 1032 or 1152, times the sub-block's scale (or a sixteenth
// of it): (n - 8) sc, exact (at most 8 * 63). Per sub-block 8 d sc - dmin m is the factor of its sum of
// x, rounded once (both products are exact in fp32).
struct WQ4K {
  static constexpr int BYTES = 144, NF = 1;  // NF: accumulators (MFMAs) per chunk
  static constexpr bool MINS = true, SWAP = true;
  struct Raw { uint4 h, q0, q1; };
  struct Scale { fh2 sl, sh; float mlo, mhi; };

  // the first of four consecutive values of half h (values 0..3 or 4..7) of chunk (q, m); the
  // chunk takes them in the order 0, 2, 1, 3 (SWAP)
  __device__ static int xoff4(int q, int m, int h) { return 64 * q + 32 * h + 4 * m; }

  __device__ static void load(const uint8_t *blk, int q, Raw &r) {
    r.h = ldw16(blk);
    r.q0 = ldw16(blk + 16 + 32 * q);
    r.q1 = ldw16(blk + 32 + 32 * q);
  }

  __device__ static Scale scale(const Raw &r, int q) {
    const uint4 h = r.h;
    const int k = 16 * (q & 1);
    // get_scale_min_k4 (src/Quants.cs:321-330) for sub-blocks 2q, 2q + 1
    const uint32_t S = q < 2 ? (h.y & 0x3F3F3F3Fu) : ((h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u));
    const uint32_t M = q < 2 ? (h.z & 0x3F3F3F3Fu) : (((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u));
    const float sclo = (float)((S >> k) & 0xFF), schi = (float)((S >> (k + 8)) & 0xFF);
    const float mlo = (float)((M >> k) & 0xFF), mhi = (float)((M >> (k + 8)) & 0xFF);
    const float dv = d(r), dm = half_hi(r.h.x);
    const _Float16 a = (_Float16)sclo, b = (_Float16)(schi * 0.0625f);
    return Scale{fh2{a, a}, fh2{b, b}, __builtin_fmaf(8.f * sclo, dv, -(dm * mlo)),
                 __builtin_fmaf(8.f * schi, dv, -(dm * mhi))};
  }

  __device__ static void frag(const Raw &r, const Scale &s, int, int m, fh8 (&f)[1]) {
    const uint32_t qd[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
    const uint32_t D = qd[m], D8 = D >> 8;
    // 1024 + n - 1032 and 1024 + 16 n - 1152
    const fh2 L = {(_Float16)-1032.f, (_Float16)-1032.f}, H = {(_Float16)-1152.f, (_Float16)-1152.f};
    const fh2 p0 = (as_fh2((D & 0x000F000Fu) | 0x64006400u) + L) * s.sl;
    const fh2 p1 = (as_fh2((D8 & 0x000F000Fu) | 0x64006400u) + L) * s.sl;
    const fh2 p2 = (as_fh2((D & 0x00F000F0u) | 0x64006400u) + H) * s.sh;
    const fh2 p3 = (as_fh2((D8 & 0x00F000F0u) | 0x64006400u) + H) * s.sh;
    f[0] = fh8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  }
  __device__ static float d(const Raw &r) { return half_lo(r.h.x); }
};

// ------------------------------------------------------------------------------------ Q6_K
// Quarter q = 2hh + ih of a super-block: half hh (128 values), i in [16 ih, 16 ih + 16) of its
// four 32-value groups g, whose 6-bit values are ql[64hh + i] (g 0, 2: low, high nibble) or
// ql[64hh + 32 + i] (g 1, 3) with bits 2g..2g+1 of qh[32hh + i], scale sc[8hh + ih + 2g]
// (src/Quants.cs:373-395). MFMA m = 2g + p takes values 128hh + 32g + 16ih + 8p + 0..7 in order;
// each byte pair becomes (1024 + q) halves by one byte permute, then two packed FMAs give
// (q - 32) sl and (q - 32) sh, sc = 16 sh + sl, for the two accumulators.
struct WQ6K {
  static constexpr int BYTES = 210, NF = 2;
  static constexpr bool MINS = false;
  // sc: the half's 8 scales; every field starts at the block's own offset within a dword
  struct Raw { uint32_t l1[5], l2[5], qh[5], sc[3], dw, sh; };
  struct Scale {};

  __device__ static int xoff4(int q, int m, int h) {
    return 128 * (q >> 1) + 32 * (m >> 1) + 16 * (q & 1) + 8 * (m & 1) + 4 * h;
  }
  static constexpr bool SWAP = false;

  template <int N>
  __device__ static void window(gu32 *a, uint32_t (&o)[N]) {
    if constexpr (N == 5) {
      const u32x4a4_t v = *reinterpret_cast<gu32x4 *>(a);
      o[0] = v.x;
      o[1] = v.y;
      o[2] = v.z;
      o[3] = v.w;
      o[4] = ldw4(a + 4);
    } else {
      ldw12(a, o);
    }
  }
  __device__ static void load(const uint8_t *blk, int q, Raw &r) {
    const int hh = q >> 1, ih = q & 1;
    gu32 *a = align4_down(blk);
    window(a + 16 * hh + 4 * ih, r.l1);
    window(a + 16 * hh + 8 + 4 * ih, r.l2);
    window(a + 32 + 8 * hh + 4 * ih, r.qh);
    window(a + 48 + 2 * hh, r.sc);
    r.dw = ldw4(a + 52);  // d: low half (block at 0 mod 4) or high half (2 mod 4)
    r.sh = misalign4(blk) * 8;
  }
  // dword i of a field's window
  template <int N>
  __device__ static uint32_t dw(const uint32_t (&w)[N], int i, uint32_t sh) {
    return __builtin_amdgcn_alignbit(w[i + 1], w[i], sh);
  }
  __device__ static Scale scale(const Raw &, int) { return Scale{}; }

  __device__ static void frag(const Raw &r, const Scale &, int q, int m, fh8 (&f)[2]) {
    const int ih = q & 1, g = m >> 1, p = m & 1;
    const uint32_t sw = dw(r.sc, g >> 1, r.sh);
    const int sc = (int)(int8_t)(sw >> (8 * (ih + 2 * (g & 1))));
    const int sl = sc & 15, shv = sc >> 4;
    const _Float16 a = (_Float16)(float)sl, na = (_Float16)(float)(-1056 * sl);
    const _Float16 b = (_Float16)(float)shv, nb = (_Float16)(float)(-1056 * shv);
    const fh2 SL = {a, a}, NL = {na, na}, SH = {b, b}, NH = {nb, nb};
    fh2 wl[4], wh[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t L = (g & 1) ? dw(r.l2, 2 * p + i, r.sh) : dw(r.l1, 2 * p + i, r.sh), H = dw(r.qh, 2 * p + i, r.sh);
      // the four 6-bit values of bytes 4i..4i+3 (src/Quants.cs:384-387)
      uint32_t v;
      if (g == 0) v = (L & 0x0F0F0F0Fu) | ((H << 4) & 0x30303030u);
      else if (g == 1) v = (L & 0x0F0F0F0Fu) | ((H << 2) & 0x30303030u);
      else if (g == 2) v = ((L >> 4) & 0x0F0F0F0Fu) | (H & 0x30303030u);
      else v = ((L >> 4) & 0x0F0F0F0Fu) | ((H >> 2) & 0x30303030u);
      // (1024 + q) halves of bytes (0, 1) and (2, 3)
      const fh2 p0 = as_fh2(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
      const fh2 p1 = as_fh2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
      wl[2 * i] = __builtin_elementwise_fma(p0, SL, NL);
      wl[2 * i + 1] = __builtin_elementwise_fma(p1, SL, NL);
      wh[2 * i] = __builtin_elementwise_fma(p0, SH, NH);
      wh[2 * i + 1] = __builtin_elementwise_fma(p1, SH, NH);
    }
    f[0] = fh8{wl[0][0], wl[0][1], wl[1][0], wl[1][1], wl[2][0], wl[2][1], wl[3][0], wl[3][1]};
    f[1] = fh8{wh[0][0], wh[0][1], wh[1][0], wh[1][1], wh[2][0], wh[2][1], wh[3][0], wh[3][1]};
  }
  __device__ static float d(const Raw &r) { return half_lo(r.dw >> r.sh); }
};

}  // namespace wl
