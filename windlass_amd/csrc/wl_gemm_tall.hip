// wl_gemm_tall.hip - prefill GEMM for prompts of more than 128 tokens over Q8_0, Q4_K, Q5_K, Q6_K and
// IQ4_XS rows (the batch branch of Transformer.MatMul, src/Transformer.cs:526-536: DecodeRow of a tile
// of weight rows, then FastMath.Block, src/FastMath.cs:216-264), on the bf16 matrix cores.
//
// A workgroup of four waves owns 128 weight rows x 512 or 256 tokens of y (JJ = 4 or 2 blocks of 32
// tokens a wave); a wave owns all 128 rows of its tokens, so its accumulators (4 x JJ tiles of
// 32 x 32) stay in AGPRs for the whole K range and one wave runs per SIMD. 256-token tiles are for
// prompts that would leave much of a 512-token tile empty (28672 x 8192 Q4_K at 200 tokens: 197 us in
// one partly filled 512-token tile, 133 in a 256-token one). K advances in steps of 32:
//   - the 128 x 32 weights of the step are decoded once per workgroup (each thread decodes 16
//     values of one row with the reference DecodeRow's fp32 operations, rounds them to bf16 and
//     writes them to LDS, a ring of four), and every wave reads the A operands of its
//     32 x 32 x 16 products from there;
//   - the tokens' B operands never pass through LDS: x is rounded to bf16 once per call into
//     fragment order (32 tokens x 32 columns = 2 x 64 lanes x 16 bytes, contiguous), so each
//     wave loads its own 2 JJ fragments per step with coalesced 1 KB reads straight into
//     registers, one step ahead.
// Formats other than Q4_K and Q6_K ran on 256-token tiles staged through LDS (gemm_kernel):
// 28672 x 8192 at 512 tokens Q8_0 553 -> 239 us, IQ4_XS 531 -> 216, Q5_K 528 -> 219. Matrices that
// share x are one launch: a 70B layer's q, k and v at 512 tokens 160 us in three with
// their sums, 110 together.
// LDS traffic per step is the decoded tile written once and read by four waves (40 KB) against
// 8 JJ MFMA per wave, and one barrier per step separates a buffer's writes
// from its reads. v_mfma_f32_32x32x16_bf16 issues at about 1.9 PFLOP/s on a whole MI355X where
// the 16 x 16 x 32 form stops at about 1.3 (measured with independent accumulator chains).
//
// Workgroups are numbered so that those sharing a K-chunk and token tile run on the same XCD
// (the dispatcher deals workgroup i to XCD i % 8), where that slice of x stays in one L2.
//
// MFMA operand layout (v_mfma_f32_32x32x16_bf16, checked on the device): lane l holds
// A[row l%32][k 8(l/32) .. +7] and B[k 8(l/32) .. +7][col l%32]; result value q of lane l is
// D[row 8(q/4) + 4(l/32) + q%4][col l%32].
#include "wl_gemm.h"

#include "wl_codecs.h"
#include "wl_frag.h"
#include "wl_gemv_impl.h"

#include "wl_device.h"

#pragma clang fp contract(off)

namespace wl {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int RM = 128;        // weight rows per workgroup
constexpr int TK = 32;         // K per step
constexpr int TLDK = TK + 8;   // padded LDS row: 80 bytes, the 16-byte reads of 8 rows cover the banks once
constexpr int TMAXS = 8;       // K-chunks at most

__device__ __forceinline__ uint32_t pk2(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  bf16x2_t v;
  v.x = (__bf16)a;  // round to nearest even (v_cvt_pk_bf16_f32)
  v.y = (__bf16)b;
  return __builtin_bit_cast(uint32_t, v);
}

// acc += A * B on the matrix cores with acc held in AGPRs (destination = accumulator operand).
// Through the builtin, the register allocator moves the accumulators between AGPRs and VGPRs at
// every step of the unrolled loop (about 47 copies per step). The compiler does not insert the
// wait states around inline assembly that an MFMA's accumulator needs, so every write of the
// accumulators before the first product and every read after the last one is separated from
// the products by mfma_drain(), with agpr_pin() holding the writes before it and the reads after.
__device__ __forceinline__ void mfma_acc(f32x16_t &acc, const uint4 &a, const uint4 &b) {
  const u32x4_t av = __builtin_bit_cast(u32x4_t, a), bv = __builtin_bit_cast(u32x4_t, b);
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(av), "v"(bv));
}

// The accumulator as it stands at this point of the program (an opaque use and redefinition):
// zeros cannot be materialized after it, nor reads hoisted before it.
__device__ __forceinline__ void agpr_pin(f32x16_t &acc) { asm volatile("" : "+a"(acc)); }

// 24 wait states, more than any MFMA result needs before another instruction reads it, and
// nothing scheduled across.
__device__ __forceinline__ void mfma_drain() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// ------------------------------------------------------------------ per-format decode
// A block's 8 sub-blocks of 32 values are the 8 steps of 32 columns. Raw holds what one thread
// needs for the 4 steps of one half-block (phase PH = S / 4): its 16 values (h = which 16 of the
// 32) of each step. The decode of a step is cut into small pieces that fit between the products
// (the matrix core runs an MFMA while the wave issues about four independent VALU instructions):
// prep<S, PART> prepares step S's scale terms (PART 0) and its quants, one byte per value
// (PARTs 1..NPREP-1); value<I> is value I (0..15) in fp32 with the reference DecodeRow's
// operations.

// The quants word v, opaque to the compiler, so each value's extraction is one
// v_cvt_f32_ubyteN of the prepared word instead of a shift-and-mask of the raw bytes.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Q4_K, 144 B: d f16 | dmin f16 | scales[12] | qs[128] (src/Quants.cs:332-350). Sub-block S's
// values are the low (S even) or high (S odd) nibbles of qs[32 (S/2) .. +32].
struct TQ4K {
  static constexpr int BYTES = 144, NPREP = 3;
  struct Raw { uint4 hdr, q[2]; };
  struct Dec { float d1, nm1; uint32_t v[4]; };
  template <int PH>
  __device__ static void load(const uint8_t *blk, int h, Raw &r) {
    r.hdr = *reinterpret_cast<const uint4 *>(blk);  // blocks are 16-byte aligned
#pragma unroll
    for (int i = 0; i < 2; i++) r.q[i] = *reinterpret_cast<const uint4 *>(blk + 16 + 32 * (2 * PH + i) + 16 * h);
  }
  template <int S, int PART>
  __device__ static void prep(const Raw &r, int, Dec &o) {
    if constexpr (PART == 0) {
      const float d = half_lo(r.hdr.x), dmin = half_hi(r.hdr.x);
      const uint32_t sc[3] = {r.hdr.y, r.hdr.z, r.hdr.w};
      auto B = [&](int i) { return (sc[i >> 2] >> (8 * (i & 3))) & 0xFFu; };
      uint32_t scv, mv;  // get_scale_min_k4 of sub-block S (src/Quants.cs:322-330)
      if constexpr (S < 4) {
        scv = B(S) & 63;
        mv = B(S + 4) & 63;
      } else {
        scv = (B(S + 4) & 0xF) | ((B(S - 4) >> 6) << 4);
        mv = (B(S + 4) >> 4) | ((B(S) >> 6) << 4);
      }
      o.d1 = d * (float)scv;
      o.nm1 = -(dmin * (float)mv);
    } else {
      const uint4 q = r.q[(S / 2) & 1];
      const uint32_t qq[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 2 * (PART - 1); i < 2 * PART; i++) o.v[i] = opaque((qq[i] >> (4 * (S & 1))) & 0x0F0F0F0Fu);
    }
  }
  // d1 * q - m1 (src/Quants.cs:345-346) as one fma with the same bits: d1 = d * sc and m1 =
  // dmin * m are products of an fp16 and a 6-bit integer (at most 17 significant bits, exact in
  // fp32), so d1 * q (q < 16) is exact too and the reference's one rounding is the subtraction's,
  // the fma's. Non-finite scales give the same infinities and NaNs.
  template <int I>
  __device__ static float value(const Dec &o) {
    return __builtin_fmaf(o.d1, (float)((o.v[I / 4] >> (8 * (I % 4))) & 0xFF), o.nm1);
  }
};

// Q6_K, 210 B: ql[128] | qh[64] | scales int8[16] | d f16 (src/Quants.cs:372-396). Half n of the
// block (128 values) is steps 4n .. 4n+3; in step qq of a half, value l (0..31) is
// ((ql[64n + 32(qq&1) + l] >> 4(qq>>1)) & 15) | ((qh[32n + l] >> 2qq) & 3) << 4, minus 32, times
// d * scales[8n + 2qq + l/16]. Blocks sit at 2-byte alignment: every field offset used here is a
// multiple of 4, so all fields share the block's misalignment and come as aligned dword windows.
struct TQ6K {
  static constexpr int BYTES = 210, NPREP = 5;
  struct Raw { uint32_t l0[5], l1[5], qh[5], sc[3], dw, sh; };
  struct Dec { float ds; uint32_t v[4]; };
  template <int PH>
  __device__ static void load(const uint8_t *blk, int h, Raw &r) {
    gu32 *a = align4_down(blk);
    r.sh = misalign4(blk) * 8;
    const int o0 = (64 * PH + 16 * h) / 4, o1 = (64 * PH + 32 + 16 * h) / 4, oh = (128 + 32 * PH + 16 * h) / 4,
              os = (192 + 8 * PH) / 4;
    const u32x4a4_t a0 = *reinterpret_cast<gu32x4 *>(a + o0);
    const u32x4a4_t a1 = *reinterpret_cast<gu32x4 *>(a + o1);
    const u32x4a4_t ah = *reinterpret_cast<gu32x4 *>(a + oh);
    r.l0[0] = a0.x; r.l0[1] = a0.y; r.l0[2] = a0.z; r.l0[3] = a0.w; r.l0[4] = a[o0 + 4];
    r.l1[0] = a1.x; r.l1[1] = a1.y; r.l1[2] = a1.z; r.l1[3] = a1.w; r.l1[4] = a[o1 + 4];
    r.qh[0] = ah.x; r.qh[1] = ah.y; r.qh[2] = ah.z; r.qh[3] = ah.w; r.qh[4] = a[oh + 4];
    ldw12(a + os, r.sc);
    r.dw = a[208 / 4];
  }
  template <int S, int PART>
  __device__ static void prep(const Raw &r, int h, Dec &o) {
    constexpr int qq = S % 4;
    if constexpr (PART == 0) {
      const float d = r.sh ? half_hi(r.dw) : half_lo(r.dw);
      // scale byte 2qq + h of the half's 8
      const uint32_t scw = __builtin_amdgcn_alignbit(r.sc[qq / 2 + 1], r.sc[qq / 2], r.sh);
      o.ds = d * (float)(int8_t)(scw >> (16 * (qq & 1) + 8 * h));
    } else {
      constexpr int i = PART - 1;  // src/Quants.cs:381-392
      const uint32_t *ql = (qq & 1) ? r.l1 : r.l0;
      const uint32_t lw = __builtin_amdgcn_alignbit(ql[i + 1], ql[i], r.sh);
      const uint32_t hw = __builtin_amdgcn_alignbit(r.qh[i + 1], r.qh[i], r.sh);
      o.v[i] = opaque(((lw >> (4 * (qq >> 1))) & 0x0F0F0F0Fu) | (((hw >> (2 * qq)) & 0x03030303u) << 4));
    }
  }
  template <int I>
  __device__ static float value(const Dec &o) {
    return o.ds * (float)((int)((o.v[I / 4] >> (8 * (I % 4))) & 0xFF) - 32);
  }
};

// Q5_K, 176 B: d f16 | dmin f16 | scales[12] | qh[32] | qs[128] (src/Quants.cs:352-370): Q4_K with bit
// S of qh byte l as the fifth bit of value l of sub-block S. d1 * q is exact for q < 32 too.
struct TQ5K {
  static constexpr int BYTES = 176, NPREP = 3;
  struct Raw { TQ4K::Raw k; uint4 qh; };
  typedef TQ4K::Dec Dec;
  template <int PH>
  __device__ static void load(const uint8_t *blk, int h, Raw &r) {
    r.k.hdr = *reinterpret_cast<const uint4 *>(blk);
    r.qh = *reinterpret_cast<const uint4 *>(blk + 16 + 16 * h);
#pragma unroll
    for (int i = 0; i < 2; i++) r.k.q[i] = *reinterpret_cast<const uint4 *>(blk + 48 + 32 * (2 * PH + i) + 16 * h);
  }
  template <int S, int PART>
  __device__ static void prep(const Raw &r, int h, Dec &o) {
    if constexpr (PART == 0) {
      TQ4K::prep<S, 0>(r.k, h, o);
    } else {
      const uint4 q = r.k.q[(S / 2) & 1];
      const uint32_t qq[4] = {q.x, q.y, q.z, q.w}, qh[4] = {r.qh.x, r.qh.y, r.qh.z, r.qh.w};
#pragma unroll
      for (int i = 2 * (PART - 1); i < 2 * PART; i++)
        o.v[i] = opaque(((qq[i] >> (4 * (S & 1))) & 0x0F0F0F0Fu) | (((qh[i] >> S) & 0x01010101u) << 4));
    }
  }
  template <int I>
  __device__ static float value(const Dec &o) { return TQ4K::value<I>(o); }
};

// Signed values of one scale.
struct TSigned { float d; uint32_t v[4]; };
template <int I>
__device__ __forceinline__ float signed_value(const TSigned &o) {
  return o.d * (float)(int8_t)(o.v[I / 4] >> (8 * (I % 4)));
}

// Q8_0: eight blocks of 34 B, d f16 | int8[32] (src/Quants.cs:251-259), at 2-byte alignment: loads at that
// alignment, since here each load and shift takes a product's slot (as aligned dword windows 14336 x 4096
// at 200 tokens took 65.0 us against 60.5).
struct TQ80 {
  static constexpr int BYTES = 272, NPREP = 2;
  struct Raw { uint4 q[4]; uint32_t d[4]; };
  typedef TSigned Dec;
  template <int PH>
  __device__ static void load(const uint8_t *blk, int h, Raw &r) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint8_t *b = blk + 34 * (4 * PH + i);
      r.d[i] = ldw2(b);
      r.q[i] = ldw16_a2(b + 2 + 16 * h);
    }
  }
  template <int S, int PART>
  __device__ static void prep(const Raw &r, int, Dec &o) {
    if constexpr (PART == 0) {
      o.d = half_lo(r.d[S % 4]);
    } else {
      const uint4 q = r.q[S % 4];
      o.v[0] = opaque(q.x);
      o.v[1] = opaque(q.y);
      o.v[2] = opaque(q.z);
      o.v[3] = opaque(q.w);
    }
  }
  template <int I>
  __device__ static float value(const Dec &o) { return signed_value<I>(o); }
};

// IQ4_XS, 136 B: d f16 | scales_h u16 | scales_l[4] | qs[128] (src/IQuants.cs:60-80): the low (h = 0) or
// high nibbles of sub-block S's 16 bytes index the 16 kvalues.
struct TIQ4XS {
  static constexpr int BYTES = 136, NPREP = 5;
  struct Raw { uint2 hdr; uint4 q[4]; };
  typedef TSigned Dec;
  template <int PH>
  __device__ static void load(const uint8_t *blk, int, Raw &r) {
    r.hdr = ldw8(blk);  // blocks are 8-byte aligned
#pragma unroll
    for (int i = 0; i < 4; i++) r.q[i] = ldw16_a2(blk + 8 + 16 * (4 * PH + i));
  }
  template <int S, int PART>
  __device__ static void prep(const Raw &r, int h, Dec &o) {
    if constexpr (PART == 0) {
      const int ls = (int)(((r.hdr.y >> (4 * S)) & 0xF) | (((r.hdr.x >> (16 + 2 * S)) & 3) << 4));
      o.d = half_lo(r.hdr.x) * (float)(ls - 32);  // src/IQuants.cs:69-72
    } else {
      const uint4 q = r.q[S % 4];
      const uint32_t qq[4] = {q.x, q.y, q.z, q.w};
      o.v[PART - 1] = opaque(iq4_signed4((qq[PART - 1] >> (4 * h)) & 0x0F0F0F0Fu));
    }
  }
  template <int I>
  __device__ static float value(const Dec &o) { return signed_value<I>(o); }
};

// ------------------------------------------------------------------ x in fragment order
// xf fragment (j, s), j = token block of 32, s = step of 32 columns, is 2 x 64 lanes x 16 bytes at
// xf + (j * nsteps + s) * 128: half u (columns 16u .. 16u+15 of the step), lane l holds token
// 32j + l%32, columns 32s + 16u + 8(l/32) .. +7 as bf16 (round to nearest even). Tokens past T
// repeat token T - 1, or where a norm wrote the fragments hold any value (their results are never
// stored, and an MFMA's columns are independent).
// One workgroup per (token block j, 8 steps): the 32 tokens' 256 columns come in as 1 KB rows
// (a wave reads one row's 256 floats), go through LDS as bf16, and leave as the 8 fragments
// (j, s0 .. s0+7), 16 KB contiguous in xf.
constexpr int FRAG_ROW = 64 + 2;  // uint2 per LDS row: 256 bf16 and a 16-byte pad

// What the fragments hold: a row of x, or silu(g) * u of the FFN (SwiGlu, src/Transformer.cs:247),
// whose fp32 pass and its rounding were two more passes over memory (2,048 tokens x 14336: 83 + 26 us).
struct LoadRow {
  const float *x;
  __device__ float4 at(int64_t i) const { return reinterpret_cast<const float4 *>(x)[i]; }
};
struct LoadSilu {
  const float *g, *u;
  __device__ float4 at(int64_t i) const {
    const float4 a = reinterpret_cast<const float4 *>(g)[i], b = reinterpret_cast<const float4 *>(u)[i];
    return make_float4(silu_mul(a.x, b.x), silu_mul(a.y, b.y), silu_mul(a.z, b.z), silu_mul(a.w, b.w));
  }
};

template <class L>
__global__ __launch_bounds__(256) void to_frag_kernel(L x, int T, int cols, uint4 *__restrict__ xf) {
  __shared__ uint2 lds[32 * FRAG_ROW];
  const int nsteps = cols / TK, groups = nsteps / 8;
  const int j = blockIdx.x / groups, s0 = (blockIdx.x % groups) * 8;
  const int tid = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int r = 4 * k + (tid >> 6), c = tid & 63;
    const int t = min(32 * j + r, T - 1);
    const float4 v = x.at(((int64_t)t * cols + TK * s0) / 4 + c);
    lds[r * FRAG_ROW + c] = make_uint2(pk2(v.x, v.y), pk2(v.z, v.w));
  }
  __syncthreads();
  uint4 *o = xf + ((int64_t)j * nsteps + s0) * 128;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const int i = tid + 256 * m;  // fragment i / 128 of the 8; piece q = (i / 32) % 4, token l = i % 32
    const int f = i >> 7, q = (i >> 5) & 3, l = i & 31;
    o[i] = *reinterpret_cast<const uint4 *>(&lds[l * FRAG_ROW + 8 * f + 2 * q]);
  }
}

struct TallArgs {
  TallMat m[TALL_MAX_MATS];
  int tile0[TALL_MAX_MATS];     // a matrix's first row tile
  float *part[TALL_MAX_MATS];   // its chunk partials [S][T][rows] (null: y is written)
  int nmat, cols, T;
  int kc;           // columns per K-chunk (whole blocks)
  const uint4 *xf;
  int tiles_m, tiles_n, nwg, remap;
  int add;          // y += result * rs
  float rs;
};

typedef uint32_t u32x4v_t __attribute__((ext_vector_type(4)));

// The wave's view of x: a buffer resource over its own JJ token blocks (a resource and its offsets
// have 32 bits; all of xf passes 4 GiB from T * cols = 2^31 on), and the per-lane offset of a
// fragment load.
struct XView {
  __amdgpu_buffer_rsrc_t rs;
  int stride;   // bytes between token blocks: nsteps * 2048, at most 2^28 (TALL_MAX_COLS)
  int vlane;    // lane * 16
};

// Fragment (token block jj of the wave, step s, half u) into registers.
__device__ __forceinline__ uint4 x_frag(const XView &xv, int jj, int s, int u) {
  const u32x4v_t v = __builtin_amdgcn_raw_buffer_load_b128(xv.rs, xv.vlane + u * 1024, jj * xv.stride + s * 2048, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

template <class G, int JJ>
struct TallState {
  typename G::Raw raw[2];   // by phase: raw[0] steps 0-3 of a block, raw[1] steps 4-7
  typename G::Dec dec[2];   // the decode state of steps s + 2 (dec[S & 1]) and s + 3
  uint4 b[2][JJ][2];        // B fragments by step parity, token block of 32, half of the step
  uint4 af[2][2][RM / 32];  // A fragments by step parity, half of the step, row tile of 32
  f32x16_t acc[RM / 32][JJ];
};

// What a step loads for the steps after it, issued from the product slots.
struct StepMem {
  const XView *xv;
  int s;                 // this step's index in the row
  const uint16_t *ar;    // step s + 1's A tile in LDS (with the lane's offset)
  const uint8_t *wnext;  // the next block's bytes (weights of a half-block ahead), or null
};

// Product K (0..NK-1) of a step, then the work that slot carries (F = 32 / NK of the decode's pieces
// a slot: one with four token blocks, two with two):
//   slots 0 .. 2 JJ - 1   the next step's B fragment K (x_frag)
//   the 8 after those     the next step's A fragments (LDS)
//   slots 0 .. 16/F - 1   the values of step s + 2's decode
//   up to 24/F - 1        their bf16 pairs; in the second of these a half-block's weight bytes, in
//                         the last the decoded values to LDS
//   the rest              the preparation of step s + 3's decode
// A scheduling barrier after each slot keeps this order, so every v_mfma is followed by one
// memory instruction and a few independent VALU instructions, which issue while the matrix core
// works, instead of the step opening with sixteen memory instructions and no product.
template <class G, int JJ, int S, int K, bool HAS1, bool DEC2, bool DEC3, bool LAST>
__device__ __forceinline__ void step_products(TallState<G, JJ> &st, int h, float (&y)[16], uint32_t (&o)[8],
                                              uint16_t *a_out, const StepMem &mem) {
  constexpr int NR = RM / 32, NK = 2 * NR * JJ, F = 32 / NK, NB = 2 * JJ;
  static_assert(NK * F == 32 && G::NPREP <= 8 && NK >= NB + 2 * NR, "decode and load slots");
  if constexpr (K < NK) {
    constexpr int u = K / (NR * JJ), i = (K / JJ) % NR, jj = K % JJ;
    mfma_acc(st.acc[i][jj], st.af[S & 1][u][i], st.b[S & 1][jj][u]);
    if constexpr (HAS1 && K < NB) st.b[(S + 1) & 1][K >> 1][K & 1] = x_frag(*mem.xv, K >> 1, mem.s + 1, K & 1);
    if constexpr (HAS1 && K >= NB && K < NB + 2 * NR) {
      constexpr int un = (K - NB) / NR, in = (K - NB) % NR;
      st.af[(S + 1) & 1][un][in] = *reinterpret_cast<const uint4 *>(mem.ar + 32 * in * TLDK + 16 * un);
    }
    if constexpr (K == 16 / F + 1 && !LAST) {
      if constexpr (S == 1) G::template load<0>(mem.wnext, h, st.raw[0]);
      if constexpr (S == 5) G::template load<1>(mem.wnext, h, st.raw[1]);
    }
    if constexpr (DEC2 && K < 16 / F) {
      y[F * K] = G::template value<F * K>(st.dec[S & 1]);
      if constexpr (F == 2) y[F * K + 1] = G::template value<F * K + 1>(st.dec[S & 1]);
    }
    if constexpr (DEC2 && K >= 16 / F && K < 24 / F) {
#pragma unroll
      for (int n = F * K - 16; n < F * K - 16 + F; n++) o[n] = pk2(y[2 * n], y[2 * n + 1]);
    }
    if constexpr (DEC2 && K == 24 / F - 1) {  // the decoded values of step s + 2 to LDS
      uint4 *ad = reinterpret_cast<uint4 *>(a_out);
      ad[0] = make_uint4(o[0], o[1], o[2], o[3]);
      ad[1] = make_uint4(o[4], o[5], o[6], o[7]);
    }
    if constexpr (DEC3 && K >= 24 / F) {
      constexpr int S3 = (S + 3) & 7, P = F * K - 24;
      if constexpr (P < G::NPREP) G::template prep<S3, P>(st.raw[S3 / 4], h, st.dec[(S + 1) & 1]);
      if constexpr (F == 2 && P + 1 < G::NPREP) G::template prep<S3, P + 1>(st.raw[S3 / 4], h, st.dec[(S + 1) & 1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    step_products<G, JJ, S, K + 1, HAS1, DEC2, DEC3, LAST>(st, h, y, o, a_out, mem);
  }
}

// Step S (0..7) of block blk. Going in, the step's A operands are in registers (af[S & 1]), its B
// operands are loaded or in flight (b[S & 1]), and the decode state of step s + 2 is ready
// (dec[S & 1]). Between its products the step loads the next step's B fragments and A operands
// (from LDS buffer (S + 1) & 3), loads the weight bytes
// of a half-block four steps ahead (at S = 1 and 5), decodes step s + 2 into buffer (S + 2) & 3
// and prepares step s + 3's decode; it ends at the barrier. Buffer (S + 1) & 3 was written
// during step s - 1 and made visible by the barrier that ended it; buffer (S + 2) & 3 held step
// s - 2's operands, read during step s - 3, so one barrier per step orders every LDS write
// against its reads.
// LAST: the row's last block (steps past its end are not prepared).
template <class G, int JJ, int S, bool LAST>
__device__ __forceinline__ void tall_step(TallState<G, JJ> &st, uint16_t (*As)[128 * TLDK], int blk,
                                          const uint8_t *wblk0, const XView &xv, int s0, int h, int aw, int ao) {
  constexpr int S1 = (S + 1) & 7, S2 = (S + 2) & 7;
  constexpr bool HAS1 = !(LAST && S == 7);  // step s + 1 exists
  constexpr bool HAS2 = !(LAST && S >= 6);  // step s + 2 exists
  constexpr bool HAS3 = !(LAST && S >= 5);  // step s + 3 exists
  StepMem mem{&xv, s0 + 8 * blk + S, As[S1 & 3] + ao, wblk0 + (blk + 1) * G::BYTES};
  float y[16];
  uint32_t o[8];
  __builtin_amdgcn_sched_barrier(0);
  step_products<G, JJ, S, 0, HAS1, HAS2, HAS3, LAST>(st, h, y, o, As[S2 & 3] + aw, mem);
  if constexpr (HAS1) __syncthreads();
}

template <class G, int JJ, bool LAST>
__device__ __forceinline__ void tall_block(TallState<G, JJ> &st, uint16_t (*As)[128 * TLDK], int blk,
                                           const uint8_t *wblk0, const XView &xv, int s0, int h, int aw, int ao) {
  tall_step<G, JJ, 0, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 1, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 2, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 3, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 4, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 5, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 6, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
  tall_step<G, JJ, 7, LAST>(st, As, blk, wblk0, xv, s0, h, aw, ao);
}

template <class G, int S, int PART>
__device__ __forceinline__ void prep_all(const typename G::Raw &r, int h, typename G::Dec &d) {
  if constexpr (PART < G::NPREP) {
    G::template prep<S, PART>(r, h, d);
    prep_all<G, S, PART + 1>(r, h, d);
  }
}

template <class G, int I>
__device__ __forceinline__ void values_all(const typename G::Dec &d, float (&y)[16]) {
  if constexpr (I < 16) {
    y[I] = G::template value<I>(d);
    values_all<G, I + 1>(d, y);
  }
}

// Decodes step S of the block whose half-block bytes are in r into LDS at ad (the prologue).
template <class G, int S>
__device__ __forceinline__ void decode_step(const typename G::Raw &r, int h, uint16_t *ad) {
  typename G::Dec d;
  prep_all<G, S, 0>(r, h, d);
  float y[16];
  values_all<G, 0>(d, y);
  uint4 *a = reinterpret_cast<uint4 *>(ad);
  a[0] = make_uint4(pk2(y[0], y[1]), pk2(y[2], y[3]), pk2(y[4], y[5]), pk2(y[6], y[7]));
  a[1] = make_uint4(pk2(y[8], y[9]), pk2(y[10], y[11]), pk2(y[12], y[13]), pk2(y[14], y[15]));
}

template <class G, int JJ>
__device__ __forceinline__ void tall_body(const TallArgs &p, const TallMat &M, float *part, uint16_t (*As)[128 * TLDK],
                                          int m0, int nt, int chunk) {
  constexpr int TWN = 32 * JJ;  // tokens per wave
  const int n0 = nt * 4 * TWN;
  const int kb = chunk * p.kc, ke = min(p.cols, kb + p.kc);
  const int nblk = (ke - kb) / 256, nsteps = p.cols / TK;
  float *y = part ? part + (int64_t)chunk * p.T * M.rows : M.y;
  const int64_t ldy = part ? M.rows : M.ldy;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);

  // decoder role: row tid / 2 of the tile, values 16h .. 16h+15 of each step (h = tid % 2). The
  // two lanes of a row read adjacent 16-byte pieces of its block, so a wave's weight load touches
  // 32 rows' lines instead of 64: the texture unit, which also carries every B fragment, spends
  // its time per line.
  const int ar = tid >> 1, h = tid & 1;
  const uint8_t *wblk0 = M.w + (int64_t)min(m0 + ar, M.rows - 1) * M.row_bytes + (int64_t)(kb / 256) * G::BYTES;
  const int aw = ar * TLDK + 16 * h;
  const int ao = (lane & 31) * TLDK + 8 * (lane >> 5);

  // this wave's JJ token blocks from jb. Where they pass the last real block (jlast), the wave loads
  // the JJ blocks ending at jlast instead and stores only its own (T > 128: there are JJ blocks).
  const int jlast = (p.T - 1) / 32, jb = (n0 + TWN * wv) / 32;
  const int jfirst = jb + JJ - 1 > jlast ? max(0, jlast - JJ + 1) : jb;
  XView xv;
  xv.stride = nsteps * 2048;
  xv.rs = __builtin_amdgcn_make_buffer_rsrc((void *)((const uint8_t *)p.xf + (int64_t)jfirst * xv.stride), (short)0,
                                            min(JJ, jlast + 1 - jfirst) * xv.stride, 0x00020000);
  xv.vlane = lane * 16;
  const int s0 = kb / TK;

  TallState<G, JJ> st;
#pragma unroll
  for (int i = 0; i < RM / 32; i++)
#pragma unroll
    for (int jj = 0; jj < JJ; jj++)
#pragma unroll
      for (int q = 0; q < 16; q++) st.acc[i][jj][q] = 0.f;
#pragma unroll
  for (int i = 0; i < RM / 32; i++)
#pragma unroll
    for (int jj = 0; jj < JJ; jj++) agpr_pin(st.acc[i][jj]);
  mfma_drain();  // the zeroed accumulators before the first product reads them

  if (nblk > 0) {
    // steps 0 and 1 decoded into buffers 0 and 1, step 2's decode prepared, step 0's operands in
    // registers
    G::template load<0>(wblk0, h, st.raw[0]);
    G::template load<1>(wblk0, h, st.raw[1]);
#pragma unroll
    for (int jj = 0; jj < JJ; jj++)
#pragma unroll
      for (int u = 0; u < 2; u++) st.b[0][jj][u] = x_frag(xv, jj, s0, u);
    decode_step<G, 0>(st.raw[0], h, As[0] + aw);
    decode_step<G, 1>(st.raw[0], h, As[1] + aw);
    prep_all<G, 2, 0>(st.raw[0], h, st.dec[0]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < RM / 32; i++)
        st.af[0][u][i] = *reinterpret_cast<const uint4 *>(As[0] + ao + 32 * i * TLDK + 16 * u);
    for (int blk = 0; blk < nblk - 1; blk++) tall_block<G, JJ, false>(st, As, blk, wblk0, xv, s0, h, aw, ao);
    tall_block<G, JJ, true>(st, As, nblk - 1, wblk0, xv, s0, h, aw, ao);
  }
  mfma_drain();
#pragma unroll
  for (int i = 0; i < RM / 32; i++)
#pragma unroll
    for (int jj = 0; jj < JJ; jj++) agpr_pin(st.acc[i][jj]);

  // value q of tile (i, jj): row 32i + 8(q/4) + 4(l/32) + q%4, token 32jj + l%32 (of the wave's tokens)
#pragma unroll
  for (int jj = 0; jj < JJ; jj++) {
    const int t = 32 * (jfirst + jj) + (lane & 31);
    const bool own = jfirst + jj >= jb;  // a block of this wave (jfirst + jj < jb + JJ always)
    if (t < p.T && own) {
#pragma unroll
      for (int i = 0; i < RM / 32; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int r0 = m0 + 32 * i + 8 * g + 4 * (lane >> 5);
          float *yp = y + (int64_t)t * ldy + r0;
          if (p.add && !part) {
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (r0 + q < M.rows) yp[q] = add_scaled(yp[q], st.acc[i][jj][4 * g + q], p.rs);
          } else if (r0 + 3 < M.rows) {
            yp[0] = st.acc[i][jj][4 * g];
            yp[1] = st.acc[i][jj][4 * g + 1];
            yp[2] = st.acc[i][jj][4 * g + 2];
            yp[3] = st.acc[i][jj][4 * g + 3];
          } else {
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (r0 + q < M.rows) yp[q] = st.acc[i][jj][4 * g + q];
          }
        }
    }
  }
}

// Token blocks of 32 a wave has: tiles of 512 (JJ = 4) or 256 tokens (JJ = 2).
template <int JJ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_tall_kernel(TallArgs p) {
  // a ring of four decoded A tiles, 128 rows each
  __shared__ __attribute__((aligned(16))) uint16_t As[4][128 * TLDK];
  const int wg = blockIdx.x;
  const int jlin = p.remap ? (wg % 8) * (p.nwg / 8) + wg / 8 : wg;
  const int mt = jlin % p.tiles_m, grp = jlin / p.tiles_m;
  const int nt = grp % p.tiles_n, chunk = grp / p.tiles_n;
  int k = 0;
  if (p.nmat > 1 && mt >= p.tile0[1]) k = 1;
  if (p.nmat > 2 && mt >= p.tile0[2]) k = 2;
  const TallMat &M = p.m[k];
  const int m0 = (mt - p.tile0[k]) * RM;
  switch (M.type) {
    case 8: tall_body<TQ80, JJ>(p, M, p.part[k], As, m0, nt, chunk); break;
    case 12: tall_body<TQ4K, JJ>(p, M, p.part[k], As, m0, nt, chunk); break;
    case 13: tall_body<TQ5K, JJ>(p, M, p.part[k], As, m0, nt, chunk); break;
    case 14: tall_body<TQ6K, JJ>(p, M, p.part[k], As, m0, nt, chunk); break;
    case 23: tall_body<TIQ4XS, JJ>(p, M, p.part[k], As, m0, nt, chunk); break;
  }
}

// y = the S chunk partials added in chunk order (y += that * rs with add). V = 4: rows, ldy and y's
// address are multiples of 4 floats, and each thread adds four adjacent outputs with 16-byte loads
// and stores. blockIdx.y: the matrix.
template <int V>
__global__ __launch_bounds__(256) void tall_combine_kernel(TallArgs p, int S) {
  typedef float fv_t __attribute__((ext_vector_type(V)));
  const TallMat &M = p.m[blockIdx.y];
  const int64_t plane = (int64_t)p.T * M.rows / V, rv = M.rows / V;
  const fv_t *pv = reinterpret_cast<const fv_t *>(p.part[blockIdx.y]);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < plane; i += (int64_t)gridDim.x * blockDim.x) {
    fv_t s = pv[i];
    for (int c = 1; c < S; c++) s += pv[c * plane + i];  // chunk order
    const int64_t t = i / rv, r = i % rv;
    fv_t *y = reinterpret_cast<fv_t *>(M.y + t * M.ldy + r * V);
    if (p.add) {
      const fv_t o = *y;
      if constexpr (V == 1) s[0] = add_scaled(o[0], s[0], p.rs);
      else
#pragma unroll
        for (int k = 0; k < V; k++) s[k] = add_scaled(o[k], s[k], p.rs);
    }
    *y = s;
  }
}

struct TallPlan {
  int jj, tiles_n, S, kc;
};

// Workgroups run one to a CU, in rounds. Both tiles are priced with every split in whole blocks: a
// block of 256 columns takes a workgroup about 6.5 us with 512-token tiles and 4.2 with 256-token ones
// (28672 x 8192 Q4_K 212 us at 512 tokens, 134 at 256; the formats with more decode, Q6_K and Q8_0, 7.0
// and 4.9: 227 / 156 and 239 / 169 us), and each K-chunk's plane is written and read once at about
// 6 TB/s. A split whose planes take more than limit bytes is left out.
TallPlan tall_plan(const TallMat *mats, int n, int cols, int T, int num_cu, int64_t limit) {
  TallPlan best{};
  double least = 0;
  int64_t tiles_m = 0, rows = 0;
  bool heavy = false;
  for (int i = 0; i < n; i++) {
    tiles_m += (mats[i].rows + RM - 1) / RM;
    rows += mats[i].rows;
    heavy = heavy || mats[i].type == 8 || mats[i].type == 14;
  }
  const int nblk = cols / 256;
  for (int jj = 4; jj >= 2; jj -= 2) {
    const double block = jj == 4 ? (heavy ? 7.0 : 6.5) : (heavy ? 4.9 : 4.2);
    const int tiles_n = (T + 128 * jj - 1) / (128 * jj);
    for (int S = 1; S <= TMAXS && S <= nblk; S++) {
      const int per = (nblk + S - 1) / S;
      if ((nblk + per - 1) / per != S) continue;  // an empty chunk
      if (S > 1 && (int64_t)S * T * rows * 4 > limit) continue;
      const int64_t rounds = (tiles_m * tiles_n * S + num_cu - 1) / num_cu;
      const double us = (double)rounds * (per * block + 3) + (S > 1 ? 4 + S * (double)T * rows * 8 / 6e6 : 0);
      if (best.jj == 0 || us < least) {
        best = TallPlan{jj, tiles_n, S, per * 256};
        least = us;
      }
    }
  }
  return best;
}

}  // namespace

bool gemm_tall_applies(int type, int T, int64_t cols) {
  return T > 128 && (type == 8 || (type >= 12 && type <= 14) || type == 23) && cols % 256 == 0 && cols <= TALL_MAX_COLS;
}

// K-chunks (of whole blocks) that give every CU a 512-token tile; one where 7/8 of the CUs have one unsplit.
static int fill_chunks(int64_t tiles, int nblk, int num_cu) {
  if (tiles * 8 >= (int64_t)num_cu * 7) return 1;
  int64_t S = (num_cu + tiles - 1) / tiles;
  S = S < TMAXS ? S : TMAXS;
  S = S < nblk ? S : nblk;
  const int64_t per = (nblk + S - 1) / S;
  return (int)((nblk + per - 1) / per);
}

int64_t tall_part_bytes(const TallMat *mats, int n, int cols, int T, int num_cu, int64_t limit) {
  int64_t rows = 0, tiles = 0;
  for (int i = 0; i < n; i++) {
    rows += mats[i].rows;
    tiles += (int64_t)((mats[i].rows + RM - 1) / RM) * ((T + 511) / 512);
  }
  auto planes = [&](int S) { return S > 1 ? (int64_t)S * T * rows * 4 : 0; };
  int S = tall_plan(mats, n, cols, T, num_cu, INT64_MAX).S;
  if (planes(S) > limit && planes(fill_chunks(tiles, cols / 256, num_cu)) <= limit)
    S = tall_plan(mats, n, cols, T, num_cu, limit).S;
  return planes(S);
}

hipError_t tall_frag_launch(const float *x, int T, int cols, void *xf, hipStream_t st) {
  hipLaunchKernelGGL(to_frag_kernel<LoadRow>, dim3((unsigned)((T + 31) / 32 * (cols / 256))), dim3(256), 0, st,
                     LoadRow{x}, T, cols, (uint4 *)xf);
  return hipGetLastError();
}

hipError_t tall_silu_frag_launch(const float *g, const float *u, int T, int cols, void *xf, hipStream_t st) {
  hipLaunchKernelGGL(to_frag_kernel<LoadSilu>, dim3((unsigned)((T + 31) / 32 * (cols / 256))), dim3(256), 0, st,
                     LoadSilu{g, u}, T, cols, (uint4 *)xf);
  return hipGetLastError();
}

hipError_t tall_matmul_launch(const TallMat *mats, int n, int cols, const void *xf, int T, bool add, float rs,
                              void *part, int64_t part_bytes, int num_cu, hipStream_t st) {
  if (n < 1 || n > TALL_MAX_MATS || cols <= 0 || !xf) return hipErrorInvalidValue;
  TallArgs a{};
  int64_t tiles = 0;
  int most = 0;
  bool v4 = true;
  for (int i = 0; i < n; i++) {
    const TallMat &m = mats[i];
    if (m.rows < 1 || !gemm_tall_applies(m.type, T, cols)) return hipErrorInvalidValue;
    a.m[i] = m;
    a.tile0[i] = (int)tiles;
    tiles += (m.rows + RM - 1) / RM;
    most = m.rows > most ? m.rows : most;
    v4 = v4 && m.rows % 4 == 0 && m.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(m.y) % 16 == 0;
  }
  const TallPlan pl = tall_plan(mats, n, cols, T, num_cu, part_bytes);  // tall_part_bytes' plan
  if (pl.S > 1 && !part) return hipErrorInvalidValue;
  float *pp = (float *)part;
  for (int i = 0; i < n; i++) {
    a.part[i] = pl.S > 1 ? pp : nullptr;
    pp += pl.S > 1 ? (int64_t)pl.S * T * mats[i].rows : 0;
  }
  a.nmat = n;
  a.cols = cols;
  a.T = T;
  a.kc = pl.kc;
  a.xf = (const uint4 *)xf;
  a.tiles_m = (int)tiles;
  a.tiles_n = pl.tiles_n;
  a.nwg = (int)tiles * pl.tiles_n * pl.S;
  a.remap = a.nwg % 8 == 0;
  a.add = add;
  a.rs = rs;
  if (pl.jj == 4) hipLaunchKernelGGL((gemm_tall_kernel<4>), dim3((unsigned)a.nwg), dim3(256), 0, st, a);
  else hipLaunchKernelGGL((gemm_tall_kernel<2>), dim3((unsigned)a.nwg), dim3(256), 0, st, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || pl.S == 1) return e;
  int64_t gc = ((int64_t)T * most / (v4 ? 4 : 1) + 255) / 256;
  if (gc > 8192) gc = 8192;
  if (v4) hipLaunchKernelGGL(tall_combine_kernel<4>, dim3((unsigned)gc, n), dim3(256), 0, st, a, pl.S);
  else hipLaunchKernelGGL(tall_combine_kernel<1>, dim3((unsigned)gc, n), dim3(256), 0, st, a, pl.S);
  return hipGetLastError();
}

}  // namespace wl
