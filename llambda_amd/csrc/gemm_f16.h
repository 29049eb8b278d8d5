// gemm_f16.h -- fp32-accurate products of split activations and packed codes on
// v_mfma_f32_16x16x32_f16, shared by the multi-token projections (gemm.hip)
// and the grouped expert products of K-quant layers (moe_f16.hip).
//
// Operands.  K runs in chunks of 256 (one Q4_K / Q6_K super-block, eight
// Q5_0 / Q8_0 blocks).  x is split as x * s = hi + lo into two f16 (11 + 11
// significant bits, |x s - hi - lo| <= 2^-23 |x s|), s the power of two that
// brings the token's largest magnitude of the chunk into [2^14, 2^15): no
// value overflows, and what subnormal lo parts lose is below 2^-39 of that
// largest value.  A weight enters as an exact f16 integer or an exact pair:
//   Q4_K        sc * q, at most 945: one f16; the chunk's d is applied once, to
//               the chunk's sums.  The sub-blocks' minima m ride in an extra
//               product per chunk, against the sub-blocks' sums of x s / 32 (hi
//               and lo).  Each add to the sums rounds in proportion to what
//               they have reached, so the hi products of a chunk run in two
//               halves (gemm_many_kernel) or four quarters (gemm_few_kernel): at
//               4096 x 4096 the error against 64 bits of N(0, 1) tokens was
//               1.36e-7 in one run, is 1.15e-7 in halves (1000 tokens) and
//               1.06e-7 in quarters (2 tokens); an fp32 evaluation has 1.2e-7.
//               The expert products (moe_f16.h) keep one run and centre the
//               codes, sc * (q - 8), with the offsets 8 sc in a second extra
//               product: as exact on such tokens, but an activation 2^13 times
//               the others leaves the rows with the smallest weights for it up
//               to eight times as far off
//   Q6_K        2^-14 sc * (q - 32), 13 bits: hi = the product rounded to f16,
//               lo = the remainder (exact); 2^14 d once per chunk (d / s alone
//               would be subnormal in chunks below 2^-99)
//   Q5_0, Q8_0  d * q, at most 18 bits, as hi + lo (exact: every product is
//               a multiple of 2^-24, f16's smallest step).  Blocks with a
//               |d| of 256 or more are multiplied in a part of their own, as
//               d / 256
// Products accumulate in fp32 over the chunk on v_mfma_f32_16x16x32_f16:
// (x hi + x lo) against one f16, or the three products hi hi + lo hi + hi lo
// against a pair (lo lo is below 2^-22 of the term).  No group's scale is
// applied outside the matrix cores, so the VALU only unpacks codes.
//
// Lane (n, g) = (lane & 15, lane >> 4) of an MFMA holds 8 codes of row n and
// 8 activations of token n; which eight of the chunk's 256 elements is free
// as long as both agree, so lane g takes the bytes that are contiguous in the
// row, and step s (0..7) takes two runs of four elements ("quads"), low and
// high, whose codes sit in one dword (K-quants: low and high nibbles) or in
// blocks 2g and 2g + 1.  Within a quad the element order is 0, 2, 1, 3: bytes
// 0 and 2 of a dword become an f16 pair of 1024 + byte by one v_perm_b32 with
// the filler byte 0x64.
#pragma once

#include "mfma.h"

namespace llhip {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float floatx4a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ floatx4 mfma_f16(const half8v& a, const half8v& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ half2v as_half2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ half2v splat2(_Float16 v) { return half2v{v, v}; }

// Bytes 0 and 2 (or 1 and 3) of v as f16 1024 + byte: one v_perm_b32 with the
// filler byte 0x64.
__device__ __forceinline__ half2v bytes02(uint32_t v) {
  return as_half2(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u));
}
__device__ __forceinline__ half2v bytes13(uint32_t v) {
  return as_half2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u));
}
// The same as f16 byte * 2^-24.
__device__ __forceinline__ half2v subnormal02(uint32_t v) {
  return as_half2(__builtin_amdgcn_perm(v, v, 0x0C020C00u));
}
__device__ __forceinline__ half2v subnormal13(uint32_t v) {
  return as_half2(__builtin_amdgcn_perm(v, v, 0x0C030C01u));
}
__device__ __forceinline__ half8v join8(half2v a, half2v b, half2v c, half2v d) {
  return half8v{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
// c * s as an exact pair hi + lo (c, s f16 whose product fits 22 bits).
__device__ __forceinline__ void exact_product(half2v c, half2v s, half2v& hi, half2v& lo) {
  hi = c * s;
  lo = __builtin_elementwise_fma(c, s, -hi);
}

// ------------------------------------------------------------ weights
// kBytes: one chunk of a row.  kPair: weights come as hi + lo.  kMin: the
// Q4_K minima product.  load(): the chunk's bytes of lane g; prepare(): its
// scales; frag(): step s's eight weights; finish(): what the chunk's sums are
// multiplied by.  quad(g, s, high): the chunk element a quad starts at; its
// inverse, for quad 16 q + l: step(l), and 256 g + 8 high as lane_bytes(l) +
// quarter_bytes(q).
template <int TYPE>
struct GemmW;

// Quads of the types whose 256 elements are 8 groups of 32: lane g takes
// groups 2g (low) and 2g + 1 (high), step s elements 4s .. 4s + 3 of each.
struct QuadsByGroup {
  static __device__ __forceinline__ int quad(int g, int s, int high) {
    return 64 * g + 32 * high + 4 * s;
  }
  static __device__ __forceinline__ int step(int l) { return l & 7; }
  static __device__ __forceinline__ int lane_bytes(int l) { return 8 * (l >> 3); }
  static constexpr int quarter_bytes(int q) { return 256 * q; }
};

// Q4_K rows: the chunk's bytes and the decode of its scales and minima.
struct Q4KRow : QuadsByGroup {
  static constexpr int kBytes = 144;
  static constexpr bool kPair = false, kMin = true, kBlocks32 = false;
  struct Raw {
    uint4 h, q0, q1;
  };
  // the 16-byte header and qs bytes [32 g, 32 g + 32); 16-byte aligned rows
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* b, uint32_t o, int g, int) {
    r.h = load16_aligned(b + o);
    const uint32_t q = o + 32u * (uint32_t)g;
    r.q0 = load16_aligned(b + q + 16);
    r.q1 = load16_aligned(b + q + 32);
  }
  // get-scale-min-k4-at (llambda.lisp:4316-4336) of sub-blocks 2g, 2g + 1
  // (both at once, in bytes 0 and 1)
  static __device__ __forceinline__ uint32_t scale_bytes(const Raw& r, int g) {
    const int shift = 8 * ((2 * g) & 3);
    const uint32_t b0 = r.h.y >> shift, b8 = r.h.w >> shift;
    return g >= 2 ? (b8 & 0x0F0Fu) | ((b0 >> 2) & 0x3030u) : b0 & 0x3F3Fu;
  }
  static __device__ __forceinline__ uint32_t min_bytes(const Raw& r, int g) {
    const int shift = 8 * ((2 * g) & 3);
    const uint32_t b4 = r.h.z >> shift, b8 = r.h.w >> shift;
    return g >= 2 ? ((b8 >> 4) & 0x0F0Fu) | ((b4 >> 2) & 0x3030u) : b4 & 0x3F3Fu;
  }
  // the minima as f16 pairs {m, m} of both sub-blocks and {m0, m1}
  static __device__ __forceinline__ void minima(uint32_t mn, uint32_t& m0, uint32_t& m1,
                                                uint32_t& m2) {
    const half2v a = splat2((_Float16)(float)(mn & 0xFFu));
    const half2v b = splat2((_Float16)(float)((mn >> 8) & 0xFFu));
    m0 = __builtin_bit_cast(uint32_t, a);
    m1 = __builtin_bit_cast(uint32_t, b);
    m2 = __builtin_bit_cast(uint32_t, half2v{a.x, b.x});
  }
  // the dword of step s's codes: low and high nibbles
  static __device__ __forceinline__ uint32_t codes(const Raw& r, int s) {
    const uint4 v = s < 4 ? r.q0 : r.q1;
    const int i = s & 3;
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
  }
};

template <>
struct GemmW<kQ4_K> : Q4KRow {
  static constexpr bool kCentred = false;
  struct Scale {
    half2v sl, sh;  // 2^10 sc of sub-block 2g, 2^6 sc of 2g + 1
    uint32_t mn;
  };
  struct Finish {
    uint32_t m0, m1, m2;  // against the sub-blocks' sums
    float d, dm;          // 2^14 d and -32 dmin
  };
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int g) {
    const uint32_t sc = scale_bytes(r, g);
    c.sl = splat2((_Float16)((float)(sc & 0xFFu) * 1024.f));
    c.sh = splat2((_Float16)((float)((sc >> 8) & 0xFFu) * 64.f));
    c.mn = min_bytes(r, g);
  }
  static __device__ __forceinline__ void finish(Finish& f, const Raw& r, const Scale& c, int) {
    minima(c.mn, f.m0, f.m1, f.m2);
    f.d = 16384.f * half_bits_to_float(r.h.x & 0xFFFFu);
    f.dm = -32.f * half_bits_to_float(r.h.x >> 16);
  }
  // 2^-14 sc q = (q 2^-24) (2^10 sc) = (16 q 2^-24) (2^6 sc): a nibble where it
  // lies in its byte is an f16 subnormal
  static __device__ __forceinline__ void frag(half8v& hi, half8v&, const Raw& r, const Scale& c,
                                              int s) {
    const uint32_t w = codes(r, s), lo = w & 0x0F0F0F0Fu, hg = w & 0xF0F0F0F0u;
    hi = join8(subnormal02(lo) * c.sl, subnormal13(lo) * c.sl, subnormal02(hg) * c.sh,
               subnormal13(hg) * c.sh);
  }
};

// --------------------------------------------------------- activations
// The chunk's scale of a token from its largest magnitude: s = 2^(14 - e),
// e the exponent of `top`, and 1 / s; both normal floats (s stops growing at
// 2^126, so chunks whose every value is below 2^-112 keep 2^-150 instead of
// 22 bits).  With an infinity among the values s stays small enough that no
// finite one overflows.
__device__ __forceinline__ void chunk_scale(float top, float& s, float& inv) {
  int e = (int)(__builtin_bit_cast(uint32_t, top) >> 23);
  e = min(max(e, 15), 254);
  s = __builtin_bit_cast(float, (uint32_t)(268 - e) << 23);
  inv = __builtin_bit_cast(float, (uint32_t)(e - 14) << 23);
}

// Four elements in quad order as f16 hi and lo (two dwords each).
__device__ __forceinline__ void split_quad(const floatx4& v, float s, uint2& hi, uint2& lo) {
  const float e[4] = {v.x, v.z, v.y, v.w};
  half4v h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = (_Float16)fmaf(e[i], s, 0.f);
    l[i] = (_Float16)fmaf(e[i], s, -(float)h[i]);
  }
  hi = __builtin_bit_cast(uint2, h);
  lo = __builtin_bit_cast(uint2, l);
}

// An infinite hi has no remainder (inf - inf would make it NaN).
__device__ __forceinline__ uint32_t drop_inf(uint32_t hi, uint32_t lo) {
  if ((hi & 0x7FFFu) == 0x7C00u) lo &= 0xFFFF0000u;
  if ((hi & 0x7FFF0000u) == 0x7C000000u) lo &= 0x0000FFFFu;
  return lo;
}
__device__ __forceinline__ bool infinite(float top) { return top == __builtin_inff(); }

__device__ __forceinline__ float abs_max4(float m, const floatx4& v) {
  return fmaxf(fmaxf(fmaxf(m, fabsf(v.x)), fmaxf(fabsf(v.y), fabsf(v.z))), fabsf(v.w));
}

// A Q4_K sub-block's sum of its 32 split activations over 32, in f16 parts:
// the sum of the hi parts as a pair (an exact sum but for hi parts below 64:
// 32 multiples of 2^-4 below 2^15), the sum of the lo parts as one.  The sum
// of x itself in fp32 would carry the rounding of its five levels of adds.
// A operand of lane (t, g): the pairs of sub-blocks 2g and 2g + 1, their lo
// sums, zero.
__device__ __forceinline__ float pair_sum(uint32_t h, float acc) {
  return __builtin_amdgcn_fdot2(as_half2(h), splat2((_Float16)1.f), acc, false);
}
__device__ __forceinline__ uint32_t split_sum(float sum) {
  const float v = sum * 0.03125f;
  const _Float16 h = (_Float16)v;
  const float hf = (float)h;
  const _Float16 l = (_Float16)(fabsf(hf) == __builtin_inff() ? 0.f : v - hf);
  return __builtin_bit_cast(uint32_t, half2v{h, l});
}
__device__ __forceinline__ uint16_t lo_sum(float sum) {
  return __builtin_bit_cast(uint16_t, (_Float16)(sum * 0.03125f));
}

// The chunk's sums into the totals: inv[i] = 1 / s of the tokens of D's rows,
// `sums` the Q4_K sums' operand.
template <typename W>
__device__ __forceinline__ void add_products(floatx4& tot, const floatx4& blk, const floatx4& inv,
                                             const typename W::Finish& c, const u32x4& sums) {
  if constexpr (W::kMin) {
    const half8v a = __builtin_bit_cast(half8v, sums);
    const half8v m = __builtin_bit_cast(half8v, u32x4{c.m0, c.m1, c.m2, 0u});
    const floatx4 mn = mfma_f16(a, m, floatx4{0.f, 0.f, 0.f, 0.f});
    floatx4 all = blk;
    if constexpr (W::kCentred)
      all = mfma_f16(a, __builtin_bit_cast(half8v, u32x4{c.c0, c.c1, c.c2, 0u}), blk);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      tot[i] = fmaf(inv[i], fmaf(c.d, all[i], c.dm * mn[i]), tot[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) tot[i] = fmaf(inv[i] * c.d, blk[i], tot[i]);
  }
}

}  // namespace llhip
