// gemm.hip -- multi-token dequant-fused projections on the matrix cores:
// y[t][r] = sum_k W[r][k] x[t][k] for packed rows and T >= 2 tokens, with the
// accuracy of an fp32 evaluation.
//
// (operands: gemm_f16.h)
#include "gemm_f16.h"
#include "gemv.h"

#include <algorithm>

namespace llhip {

// v_mul_u32_u24 (a plain product becomes a v_mul_lo_u32 here, at a quarter of
// the rate; written in inline asm it would get no wait states after an MFMA
// whose result lies in its register).
extern "C" __device__ uint32_t mul_u24(uint32_t a, uint32_t b) __asm("llvm.amdgcn.mul.u24.i32");

// Rows that start on any even byte: b moves down to its dword, and the dword
// at or below the old b + o is at the returned offset from it, `shift` bytes
// below.  (The offset is formed from the dword base, so it never goes below
// zero, where 32 bits would wrap.)
__device__ __forceinline__ uint32_t dword_offset(const uint8_t*& b, uint32_t o, uint32_t& shift) {
  const uint32_t low = (uint32_t)reinterpret_cast<uintptr_t>(b) & 3u;
  b -= low;
  o += low;
  shift = o & 3u;
  return o - shift;
}
// N dwords from byte b + o + shift, b + o on a dword (N + 1 are read, by
// 16-byte loads as far as they go).
template <int N>
__device__ __forceinline__ void load_dwords(uint32_t (&w)[N], const uint8_t* b, uint32_t o,
                                            uint32_t shift) {
  const uint8_t* p = b + o;
  uint32_t t[N + 1];
#pragma unroll
  for (int i = 0; i + 4 <= N + 1; i += 4) {
    const u32x4a4 v = *reinterpret_cast<const u32x4a4*>(p + 4 * i);
    t[i] = v.x;
    t[i + 1] = v.y;
    t[i + 2] = v.z;
    t[i + 3] = v.w;
  }
#pragma unroll
  for (int i = (N + 1) & ~3; i < N + 1; ++i) t[i] = *reinterpret_cast<const uint32_t*>(p + 4 * i);
#pragma unroll
  for (int i = 0; i < N; ++i) w[i] = __builtin_amdgcn_alignbyte(t[i + 1], t[i], shift);
}

// Element 128h + 32k + l: ql byte 64h + 32 (k & 1) + l (nibble k >> 1), qh
// byte 32h + l (bits 2k), scale 8h + 2k + (l >> 4) (llambda.lisp:4203-4310).
// Lane g takes h = g >> 1 and l = 16 (g & 1) .. + 15; step s = 2i + kk takes
// l = 16 (g & 1) + 4i .. + 3 of k = kk (low) and kk + 2 (high).
template <>
struct GemmW<kQ6_K> {
  static constexpr int kBytes = 210;
  static constexpr bool kPair = true, kMin = false, kBlocks32 = false;
  static __device__ __forceinline__ int quad(int g, int s, int high) {
    return 128 * (g >> 1) + 32 * ((s & 1) + 2 * high) + 16 * (g & 1) + 4 * (s >> 1);
  }
  static __device__ __forceinline__ int step(int l) { return 2 * (l & 3) + (l >> 3); }
  static __device__ __forceinline__ int lane_bytes(int l) { return 256 * ((l >> 2) & 1); }
  static constexpr int quarter_bytes(int q) { return 512 * (q >> 1) + 8 * (q & 1); }
  struct Raw {
    uint4 la, lb, qh;
    uint32_t s[2], d;  // scales 8h .. 8h + 7
  };
  struct Scale {
    half2v sc[4];  // 2^-14 sc
  };
  struct Finish {
    float d;
  };
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* b, uint32_t o, int g, int) {
    // 64 (g >> 1) + 16 (g & 1) of ql, 32 (g >> 1) + 16 (g & 1) of qh, 8 (g >> 1) of the scales
    const uint32_t h = (uint32_t)g >> 1, e = 16u * ((uint32_t)g & 1u);
    r.d = *reinterpret_cast<const uint16_t*>(b + o + 208);
    uint32_t sh;
    const uint32_t a = dword_offset(b, o, sh);
    load_dwords(reinterpret_cast<uint32_t(&)[4]>(r.la), b, a + 64 * h + e, sh);
    load_dwords(reinterpret_cast<uint32_t(&)[4]>(r.lb), b, a + 64 * h + 32 + e, sh);
    load_dwords(reinterpret_cast<uint32_t(&)[4]>(r.qh), b, a + 128 + 32 * h + e, sh);
    load_dwords(r.s, b, a + 192 + 8 * h, sh);
  }
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int g) {
    const int b = 8 * (g & 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t v = r.s[k >> 1] >> (16 * (k & 1) + b);
      c.sc[k] = splat2((_Float16)(0x1p-14f * (float)(int)(int8_t)(v & 0xFFu)));
    }
  }
  static __device__ __forceinline__ void finish(Finish& f, const Raw& r, const Scale&, int) {
    f.d = 0x1p14f * half_bits_to_float(r.d);
  }
  static __device__ __forceinline__ void frag(half8v& hi, half8v& lo, const Raw& r, const Scale& c,
                                              int s) {
    const int i = s >> 1, kk = s & 1;
    const uint4 q = kk ? r.lb : r.la;
    const uint32_t w = i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w;
    const uint32_t v = i == 0 ? r.qh.x : i == 1 ? r.qh.y : i == 2 ? r.qh.z : r.qh.w;
    const uint32_t cl = (w & 0x0F0F0F0Fu) | (((v >> (2 * kk)) & 0x03030303u) << 4);
    const uint32_t ch = ((w >> 4) & 0x0F0F0F0Fu) | (((v >> (2 * kk + 4)) & 0x03030303u) << 4);
    const half2v off = splat2((_Float16)-1056.f);
    half2v h[4], l[4];
    exact_product(bytes02(cl) + off, c.sc[kk], h[0], l[0]);
    exact_product(bytes13(cl) + off, c.sc[kk], h[1], l[1]);
    exact_product(bytes02(ch) + off, c.sc[kk + 2], h[2], l[2]);
    exact_product(bytes13(ch) + off, c.sc[kk + 2], h[3], l[3]);
    hi = join8(h[0], h[1], h[2], h[3]);
    lo = join8(l[0], l[1], l[2], l[3]);
  }
};

// Scales of a 32-block type: d of blocks 2g and 2g + 1.  Blocks past the row's
// end (the last chunk of a K that 256 does not divide) count 0.  A |d| of 256
// or more would leave f16's range in d q: a wave that meets one forms its sums
// anew in two parts, the large scales as d / 256, each with the other part's
// blocks at 0 (d / 256 of the small ones would fall among f16's subnormals).
struct BlockScale {
  half2v sl, sh;
  bool large;  // this lane has a |d| of 256 or more
  __device__ __forceinline__ void set(uint32_t d0, uint32_t d1, int g, int blocks) {
    d0 = 2 * g < blocks ? d0 & 0xFFFFu : 0u;
    d1 = 2 * g + 1 < blocks ? d1 & 0xFFFFu : 0u;
    large = is_large(d0) || is_large(d1);
    sl = as_half2(d0 | (d0 << 16));
    sh = as_half2(d1 | (d1 << 16));
  }
  __device__ __forceinline__ void set_part(bool part, uint32_t d0, uint32_t d1, int g, int blocks) {
    set(d0, d1, g, blocks);
    const half2v f = splat2((_Float16)(part ? 1.f / 256.f : 1.f));
    sl = is_large(d0) == part ? sl * f : splat2((_Float16)0.f);
    sh = is_large(d1) == part ? sh * f : splat2((_Float16)0.f);
  }
  static __device__ __forceinline__ bool is_large(uint32_t d) { return (d & 0x7FFFu) >= 0x5C00u; }
};

template <>
struct GemmW<kQ8_0> : QuadsByGroup {
  static constexpr int kBytes = 272;
  static constexpr bool kPair = true, kMin = false, kBlocks32 = true;
  struct Raw {
    uint32_t w[17];  // blocks 2g and 2g + 1, 34 bytes each
    int blocks;
  };
  typedef BlockScale Scale;
  struct Finish {
    float d;
  };
  static __device__ __forceinline__ void finish(Finish& f, const Raw&, const Scale&, int) {
    f.d = 1.f;
  }
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* b, uint32_t o, int g,
                                              int blocks) {
    uint32_t sh;
    const uint32_t a = dword_offset(b, o + 68u * (uint32_t)g, sh);
    load_dwords(r.w, b, a, sh);
    r.blocks = blocks;
  }
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int g) {
    c.set(r.w[0], r.w[8] >> 16, g, r.blocks);
  }
  static __device__ __forceinline__ void prepare_part(bool part, Scale& c, const Raw& r, int g) {
    c.set_part(part, r.w[0], r.w[8] >> 16, g, r.blocks);
  }
  static __device__ __forceinline__ void frag(half8v& hi, half8v& lo, const Raw& r, const Scale& c,
                                              int s) {
    // block 2g's codes start at byte 2, block 2g + 1's at byte 36
    const uint32_t a = __builtin_amdgcn_alignbyte(r.w[s + 1], r.w[s], 2) ^ 0x80808080u;
    const uint32_t b = r.w[9 + s] ^ 0x80808080u;
    const half2v off = splat2((_Float16)-1152.f);
    half2v h[4], l[4];
    exact_product(bytes02(a) + off, c.sl, h[0], l[0]);
    exact_product(bytes13(a) + off, c.sl, h[1], l[1]);
    exact_product(bytes02(b) + off, c.sh, h[2], l[2]);
    exact_product(bytes13(b) + off, c.sh, h[3], l[3]);
    hi = join8(h[0], h[1], h[2], h[3]);
    lo = join8(l[0], l[1], l[2], l[3]);
  }
};

template <>
struct GemmW<kQ5_0> : QuadsByGroup {
  static constexpr int kBytes = 176;
  static constexpr bool kPair = true, kMin = false, kBlocks32 = true;
  struct Raw {
    uint32_t w[11];  // blocks 2g and 2g + 1, 22 bytes each
    int blocks;
  };
  typedef BlockScale Scale;
  struct Finish {
    float d;
  };
  static __device__ __forceinline__ void finish(Finish& f, const Raw&, const Scale&, int) {
    f.d = 1.f;
  }
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* b, uint32_t o, int g,
                                              int blocks) {
    uint32_t sh;
    const uint32_t a = dword_offset(b, o + 44u * (uint32_t)g, sh);
    load_dwords(r.w, b, a, sh);
    r.blocks = blocks;
  }
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int g) {
    c.set(r.w[0], r.w[5] >> 16, g, r.blocks);
  }
  static __device__ __forceinline__ void prepare_part(bool part, Scale& c, const Raw& r, int g) {
    c.set_part(part, r.w[0], r.w[5] >> 16, g, r.blocks);
  }
  // element 4s + b: nibble s >> 2 of qs byte 4 (s & 3) + b, fifth bit 4s + b of qh
  static __device__ __forceinline__ uint32_t code(uint32_t qs, uint32_t qh, int s) {
    const uint32_t n = s < 4 ? qs & 0x0F0F0F0Fu : (qs >> 4) & 0x0F0F0F0Fu;
    const uint32_t bits = mul_u24((qh >> (4 * s)) & 0xFu, 0x204081u);  // bit i of the nibble to bit 8 i
    return n | ((bits & 0x01010101u) << 4);
  }
  static __device__ __forceinline__ void frag(half8v& hi, half8v& lo, const Raw& r, const Scale& c,
                                              int s) {
    const int i = s & 3;
    // block 2g: qh at byte 2, qs at byte 6; block 2g + 1 at byte 22: qh 24, qs 28
    const uint32_t qh = __builtin_amdgcn_alignbyte(r.w[1], r.w[0], 2);
    const uint32_t qs = __builtin_amdgcn_alignbyte(r.w[i + 2], r.w[i + 1], 2);
    const uint32_t a = code(qs, qh, s), b = code(r.w[7 + i], r.w[6], s);
    const half2v off = splat2((_Float16)-1040.f);
    half2v h[4], l[4];
    exact_product(bytes02(a) + off, c.sl, h[0], l[0]);
    exact_product(bytes13(a) + off, c.sl, h[1], l[1]);
    exact_product(bytes02(b) + off, c.sh, h[2], l[2]);
    exact_product(bytes13(b) + off, c.sh, h[3], l[3]);
    hi = join8(h[0], h[1], h[2], h[3]);
    lo = join8(l[0], l[1], l[2], l[3]);
  }
};


struct GemmArgs {
  const uint8_t* w;
  int64_t row_bytes;
  int rows, K, chunks;
  const float* x;
  int64_t x_stride;
  int tokens;
  float* y;
  int64_t y_stride;
  int row_tiles, token_tiles;  // gemm_many_kernel
};

// The activations of lane (token n, group g) in chunk c, xr the token's row:
// split into ah and al, with 1 / s of the tokens of D's rows in inv.
template <typename W>
__device__ __forceinline__ void split_tokens(half8v (&ah)[8], half8v (&al)[8], floatx4& inv,
                                             const float* xr, int c, int K, int g) {
  floatx4 v[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int k = 256 * c + W::quad(g, q >> 1, q & 1);
    v[q] = (!W::kBlocks32 || k < K) ? (floatx4)*reinterpret_cast<const floatx4a4*>(xr + k)
                                    : floatx4{0.f, 0.f, 0.f, 0.f};
  }
  float top = 0.f;
#pragma unroll
  for (int q = 0; q < 16; ++q) top = abs_max4(top, v[q]);
  top = fmaxf(top, __shfl_xor(top, 16));
  top = fmaxf(top, __shfl_xor(top, 32));
  float s, inv1;
  chunk_scale(top, s, inv1);
  const bool special = __any(infinite(top));
#pragma unroll
  for (int st = 0; st < 8; ++st) {
    uint2 h0, l0, h1, l1;
    split_quad(v[2 * st], s, h0, l0);
    split_quad(v[2 * st + 1], s, h1, l1);
    ah[st] = __builtin_bit_cast(half8v, u32x4{h0.x, h0.y, h1.x, h1.y});
    al[st] = __builtin_bit_cast(half8v, u32x4{l0.x, l0.y, l1.x, l1.y});
  }
  if (special) {
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const u32x4 h = __builtin_bit_cast(u32x4, ah[st]);
      u32x4 l = __builtin_bit_cast(u32x4, al[st]);
#pragma unroll
      for (int i = 0; i < 4; ++i) l[i] = drop_inf(h[i], l[i]);
      al[st] = __builtin_bit_cast(half8v, l);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) inv[i] = __shfl(inv1, 4 * g + i);
}

// A wave's sums of RT row tiles and JT token tiles over chunks first, first +
// step, ... in two parts (BlockScale), its operands straight from memory.  Rows
// without a large scale keep their sums in the large part (0 times x).
template <typename W, int RT, int JT>
__device__ __forceinline__ void sum_in_parts(floatx4 (&tot)[RT][JT], const GemmArgs& a,
                                             const uint8_t* wbase, const uint32_t (&woff)[RT],
                                             int tok0, int first, int step, int lane) {
  const int n = lane & 15, g = lane >> 4;
#pragma unroll 1
  for (int j = 0; j < JT; ++j) {
    const float* xr = a.x + (int64_t)min(tok0 + 16 * j + n, a.tokens - 1) * a.x_stride;
    floatx4 sum[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) sum[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = first; c < a.chunks; c += step) {
      half8v ah[8], al[8];
      floatx4 inv;
      split_tokens<W>(ah, al, inv, xr, c, a.K, g);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        typename W::Raw raw;
        W::load(raw, wbase + (uint32_t)c * (uint32_t)W::kBytes, woff[r], g,
                min(8, (a.K >> 5) - 8 * c));
#pragma unroll 1
        for (int part = 0; part < 2; ++part) {
          typename W::Scale sc;
          W::prepare_part(part, sc, raw, g);
          floatx4 blk = {0.f, 0.f, 0.f, 0.f};
          half8v bh[8], bl;
#pragma unroll
          for (int st = 0; st < 8; ++st) {
            W::frag(bh[st], bl, raw, sc, st);
            blk = mfma_f16(al[st], bh[st], blk);
            blk = mfma_f16(ah[st], bl, blk);
          }
#pragma unroll
          for (int st = 0; st < 8; ++st) blk = mfma_f16(ah[st], bh[st], blk);
          const uint64_t m = __ballot(sc.large);
          const uint32_t rows = (uint32_t)(m | (m >> 16) | (m >> 32) | (m >> 48));
          if (part == 0 || ((rows >> n) & 1u)) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              sum[r][i] = fmaf(part ? 256.f * inv[i] : inv[i], blk[i], sum[r][i]);
          }
        }
      }
    }
    // tile j's sums end up in tot[.][j] after the last turn
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int i = 0; i + 1 < JT; ++i) tot[r][i] = tot[r][i + 1];
      tot[r][JT - 1] = sum[r];
    }
  }
}

// --------------------------------------------------------- few tokens
// One token tile of 16 per workgroup column; the workgroup's KW waves share
// 16 RT rows and deal the chunks among themselves, each wave holding its
// chunk's activations in registers (lane (t, g) loads, scales and splits the
// 64 elements its own operand slots need: no LDS, no barrier before the
// waves' sums meet).  7 tokens through Q4_K 14336 x 4096 take 14.9 us (2.2
// TB/s; 186 us when each four tokens read the rows again and the VALU formed
// the products).  There the VALU issues for 40% of the SIMD cycles (splitting
// x and unpacking) and the matrix cores work for 11%; the rest is latency:
// nothing of a wave's next chunk is requested before this one is done.
template <int TYPE, int RT, int KW>
__global__ void __launch_bounds__(64 * KW)
gemm_few_kernel(GemmArgs a) {
  using W = GemmW<TYPE>;
  __shared__ floatx4 red[KW > 1 ? KW - 1 : 1][RT][64];
  // the wave's number is uniform: so are the loop over its chunks and their bases
  const int lane = threadIdx.x & 63, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16 * RT, tok0 = blockIdx.y * 16;
  const float* xr = a.x + (int64_t)min(tok0 + n, a.tokens - 1) * a.x_stride;
  const uint8_t* wbase = a.w + (int64_t)row0 * a.row_bytes;
  uint32_t woff[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    woff[r] = (uint32_t)(min(row0 + 16 * r + n, a.rows - 1) - row0) * (uint32_t)a.row_bytes;
  floatx4 tot[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) tot[r] = floatx4{0.f, 0.f, 0.f, 0.f};
  bool large = false;  // 32-block types: a large scale among this lane's

  for (int c = kw; c < a.chunks; c += KW) {
    const int blocks = W::kBlocks32 ? min(8, (a.K >> 5) - 8 * c) : 8;
    floatx4 v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int k = 256 * c + W::quad(g, q >> 1, q & 1);
      v[q] = (!W::kBlocks32 || k < a.K)
                 ? (floatx4)*reinterpret_cast<const floatx4a4*>(xr + k)
                 : floatx4{0.f, 0.f, 0.f, 0.f};
    }
    typename W::Raw raw[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
      W::load(raw[r], wbase + (uint32_t)c * (uint32_t)W::kBytes, woff[r], g, blocks);

    float top = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) top = abs_max4(top, v[q]);
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    float s, inv1;
    chunk_scale(top, s, inv1);
    half8v ah[8], al[8];
    const bool special = __any(infinite(top));
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      uint2 h0, l0, h1, l1;
      split_quad(v[2 * st], s, h0, l0);
      split_quad(v[2 * st + 1], s, h1, l1);
      ah[st] = __builtin_bit_cast(half8v, u32x4{h0.x, h0.y, h1.x, h1.y});
      al[st] = __builtin_bit_cast(half8v, u32x4{l0.x, l0.y, l1.x, l1.y});
    }
    if (special) {
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        const u32x4 h = __builtin_bit_cast(u32x4, ah[st]);
        u32x4 l = __builtin_bit_cast(u32x4, al[st]);
#pragma unroll
        for (int i = 0; i < 4; ++i) l[i] = drop_inf(h[i], l[i]);
        al[st] = __builtin_bit_cast(half8v, l);
      }
    }
    u32x4 sums = {0u, 0u, 0u, 0u};
    if constexpr (W::kMin) {
      float h[2] = {0.f, 0.f}, l[2] = {0.f, 0.f};
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        const u32x4 hv = __builtin_bit_cast(u32x4, ah[st]), lv = __builtin_bit_cast(u32x4, al[st]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          h[i >> 1] = pair_sum(hv[i], h[i >> 1]);
          l[i >> 1] = pair_sum(lv[i], l[i >> 1]);
        }
      }
      sums = u32x4{split_sum(h[0]), split_sum(h[1]),
                   (uint32_t)lo_sum(l[0]) | ((uint32_t)lo_sum(l[1]) << 16), 0u};
    }
    floatx4 inv;
#pragma unroll
    for (int i = 0; i < 4; ++i) inv[i] = __shfl(inv1, 4 * g + i);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      typename W::Scale sc;
      W::prepare(sc, raw[r], g);
      if constexpr (W::kBlocks32) large |= sc.large;
      // the small products first: each add to the sums rounds in proportion
      // to what they have reached
      floatx4 blk = {0.f, 0.f, 0.f, 0.f};
      half8v bh[8], bl;
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        W::frag(bh[st], bl, raw[r], sc, st);
        blk = mfma_f16(al[st], bh[st], blk);
        if constexpr (W::kPair) blk = mfma_f16(ah[st], bl, blk);
      }
      if constexpr (W::kMin) {
        // in quarters: their chains run side by side
        floatx4 part[4];
#pragma unroll
        for (int st = 0; st < 8; ++st)
          part[st >> 1] = mfma_f16(ah[st], bh[st], st & 1 ? part[st >> 1] : floatx4{0.f, 0.f, 0.f, 0.f});
        blk += (part[0] + part[1]) + (part[2] + part[3]);
      } else {
#pragma unroll
        for (int st = 0; st < 8; ++st) blk = mfma_f16(ah[st], bh[st], blk);
      }
      typename W::Finish fin;
      W::finish(fin, raw[r], sc, g);
      add_products<W>(tot[r], blk, inv, fin, sums);
    }
  }
  if constexpr (W::kBlocks32) {
    // (out of the loop above, which runs 2 to 5% longer with that branch or the
    // parts' selects in it)
    if (__any(large)) [[unlikely]]
      sum_in_parts<W, RT, 1>(reinterpret_cast<floatx4(&)[RT][1]>(tot), a, wbase, woff, tok0, kw, KW, lane);
  }
  if constexpr (KW > 1) {
    if (kw > 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r) red[kw - 1][r][lane] = tot[r];
    }
    __syncthreads();
    if (kw != 0) return;
    // the first wave adds them, in wave order
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < KW - 1; ++q) tot[r] += red[q][r][lane];
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = row0 + 16 * r + n;
    if (row < a.rows)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = tok0 + 4 * g + i;
        if (t < a.tokens) a.y[(int64_t)t * a.y_stride + row] = tot[r][i];
      }
  }
}

// Sums of V (4 or 8) values over aligned groups of eight lanes; lane i of a
// group receives the sum of value i (i % 4 for V = 4).  b2, b1, b0: bits of i.
template <int V>
__device__ __forceinline__ float scatter_sum(const float* v, bool b2, bool b1, bool b0) {
  float r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (V == 8)
      r[k] = (b2 ? v[k + 4] : v[k]) + dpp<kDppHalfMirror>(b2 ? v[k] : v[k + 4]);
    else
      r[k] = v[k] + dpp<kDppHalfMirror>(v[k]);
  }
  float u[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) u[k] = (b1 ? r[k + 2] : r[k]) + dpp<kDppXor2>(b1 ? r[k] : r[k + 2]);
  return (b0 ? u[1] : u[0]) + dpp<kDppXor1>(b0 ? u[0] : u[1]);
}

// --------------------------------------------------------- many tokens
// RW waves of 16 RT rows each share the split activations of 16 JT tokens in
// LDS; KW such groups deal the chunks among themselves.  Two chunks' images
// take turns: the next chunk's activations are requested before this chunk's
// products and split after them, so a chunk costs one barrier and its memory
// round trips run beside the products; the next chunk's weights go straight
// from memory into registers.  A load instruction covers 64 elements of four
// tokens (256 contiguous bytes each), the token's largest magnitude meets over
// 16 lanes, and the operand image is [token tile][step][hi, lo][16 bytes per
// lane], lane positions XORed with the step so that the writes of one
// instruction spread over the banks.
// Measured, card to card: 2048 tokens through Q4_K 14336 x 4096 0.63 to 0.70 ms
// (340 to 380 TFLOP/s; 49.8 ms in passes of four tokens on the VALU), 1000
// tokens through Q6_K 4096 x 14336 0.40 to 0.45 ms (31.7), 129 through Q8_0
// 1024 x 2688 14.6 us (517).  Bound by
// instruction issue: of the SIMD cycles of the first the VALU takes 47% (5.4
// instructions per MFMA: unpacking, splitting, adding the chunks' sums) and
// the matrix cores 35, of the second 38 and 38.
template <int TYPE, int JT>
struct GemmLds {
  static constexpr int kX = JT * 16384;             // split activations
  static constexpr int kInv = kX;                   // 1 / s per token
  static constexpr int kSums = kInv + JT * 64;      // Q4_K: the sums' operands
  static constexpr int kBytes = kSums + (GemmW<TYPE>::kMin ? JT * 1024 : 0);
};

template <int TYPE, int RT, int JT, int RW, int KW>
__global__ void __launch_bounds__(64 * RW * KW, 2)
gemm_many_kernel(GemmArgs a) {
  using W = GemmW<TYPE>;
  using L = GemmLds<TYPE, JT>;
  constexpr int P = 4 * JT / RW;  // groups of four tokens a wave splits
  static_assert(P * RW == 4 * JT, "token groups");
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rw = wave % RW, kw = wave / RW;
  const int n = lane & 15, g = lane >> 4;
  uint8_t* lds = smem + kw * 2 * L::kBytes;

  // Workgroup b runs on XCD b % 8: each XCD takes one contiguous run of
  // tiles, in groups of 8 row tiles by all token tiles, so that the tiles in
  // flight on an XCD share rows and tokens in its L2.
  const int total = a.row_tiles * a.token_tiles, per = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= total || (int)(blockIdx.x >> 3) >= per) return;
  const int band = tile / (8 * a.token_tiles), rest = tile - band * 8 * a.token_tiles;
  const int band_rows = min(8, a.row_tiles - 8 * band);
  const int tt = rest / band_rows, rt = 8 * band + (rest - tt * band_rows);
  const int row0 = (rt * RW + rw) * 16 * RT, tok0 = tt * 16 * JT;

  // uniform bases and 32-bit lane offsets (gemm_launch bounds the strides)
  const int rbase = __builtin_amdgcn_readfirstlane(min(row0, a.rows - 1));
  const uint8_t* wbase = a.w + (int64_t)rbase * a.row_bytes;
  uint32_t woff[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    woff[r] = (uint32_t)(min(row0 + 16 * r + n, a.rows - 1) - rbase) * (uint32_t)a.row_bytes;
  const float* xbase = a.x + (int64_t)tok0 * a.x_stride;
  uint32_t xoff[P];
#pragma unroll
  for (int p = 0; p < P; ++p)
    xoff[p] = 4 * ((uint32_t)(min(tok0 + 4 * (P * rw + p) + g, a.tokens - 1) - tok0) *
                       (uint32_t)a.x_stride + 4 * n);

  floatx4 tot[RT][JT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < JT; ++j) tot[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  typename W::Raw raw[RT];
  auto load_rows = [&](int c) {
    const int blocks = W::kBlocks32 ? min(8, (a.K >> 5) - 8 * c) : 8;
#pragma unroll
    for (int r = 0; r < RT; ++r)
      W::load(raw[r], wbase + (uint32_t)c * (uint32_t)W::kBytes, woff[r], g, blocks);
  };
  // v[p][q]: token 4 (P rw + p) + g, elements 64 q + 4 n .. + 3
  floatx4 v[P][4];
  auto load_x = [&](int c) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[p][q] = (!W::kBlocks32 || 256 * c + 64 * q + 4 * n < a.K)
                      ? (floatx4)*reinterpret_cast<const floatx4a4*>(
                            reinterpret_cast<const uint8_t*>(xbase + 256 * c + 64 * q) + xoff[p])
                      : floatx4{0.f, 0.f, 0.f, 0.f};
  };
  auto split_x = [&](uint8_t* buf) {
    const int own = (int)opaque((uint32_t)lane);  // addresses not kept over the products
    const int n = own & 15, g = own >> 4;
    float top[P], most = 0.f;
    float hs[W::kMin ? 4 * P : 1], ls[W::kMin ? 4 * P : 1];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float m = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) m = abs_max4(m, v[p][q]);
      m = fmaxf(m, dpp<kDppXor1>(m));
      m = fmaxf(m, dpp<kDppXor2>(m));
      m = fmaxf(m, dpp<kDppHalfMirror>(m));
      top[p] = fmaxf(m, dpp<kDppMirror>(m));
      most = fmaxf(most, top[p]);
    }
    const int step = W::step(n);
    uint8_t* lane_at = buf + 2048 * step + W::lane_bytes(n);
    // the group's first token is token t of the workgroup's
    auto image = [&](int t) {
      return lane_at + 16384 * (t >> 4) + 128 * ((t >> 3) & 1) + 16 * (((t & 4) + g) ^ step);
    };
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float s, inv;
      chunk_scale(top[p], s, inv);
      const int t = 4 * (P * rw + p);
      uint8_t* at = image(t);
      reinterpret_cast<float*>(buf + L::kInv)[t + g] = inv;  // 16 lanes, one value
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint2 hi, lo;
        split_quad(v[p][q], s, hi, lo);
        *reinterpret_cast<uint2*>(at + W::quarter_bytes(q)) = hi;
        *reinterpret_cast<uint2*>(at + W::quarter_bytes(q) + 1024) = lo;
        if constexpr (W::kMin) {
          hs[4 * p + q] = pair_sum(hi.y, pair_sum(hi.x, 0.f));
          ls[4 * p + q] = pair_sum(lo.y, pair_sum(lo.x, 0.f));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (W::kMin) {
      // sub-block 2q + (n >> 3) of token t + g: sums over eight lanes, lane n & 7
      // taking value n & 7 of the eight (p, q) of two token groups
      constexpr int V = 4 * P < 8 ? 4 * P : 8;
      const bool b2 = n & 4, b1 = n & 2, b0 = n & 1;
#pragma unroll
      for (int at = 0; at < 4 * P; at += V) {
        const float h = scatter_sum<V>(hs + at, b2, b1, b0), l = scatter_sum<V>(ls + at, b2, b1, b0);
        const int i = at + (n & (V - 1)), t = 4 * (P * rw + (i >> 2));
        uint8_t* to = buf + L::kSums + 1024 * (t >> 4) + 16 * ((t & 15) + g + 16 * (i & 3));
        *reinterpret_cast<uint32_t*>(to + 4 * (n >> 3)) = split_sum(h);
        *reinterpret_cast<uint16_t*>(to + 8 + 2 * (n >> 3)) = lo_sum(fabsf(h) == __builtin_inff() ? 0.f : l);
      }
    }
    if (__any(infinite(most))) {
      // an infinity has no remainder (inf - inf made it NaN)
#pragma unroll
      for (int p = 0; p < P; ++p) {
        uint8_t* at = image(4 * (P * rw + p)) + 1024;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (infinite(fabsf(v[p][q][e])))
              *reinterpret_cast<uint16_t*>(at + W::quarter_bytes(q) + 4 * (e & 1) + (e & 2)) = 0;
      }
    }
  };

  // y = tot, or y += tot with every y requested before the first add (the
  // addresses are formed here each time: kept over the chunks they cost the
  // products their registers)
  auto store_rows = [&](bool add) {
    const int at = (int)opaque((uint32_t)lane);
    const int left = a.rows - row0 - (at & 15), t0 = tok0 + 4 * (at >> 4);
    float* y0 = a.y + (int64_t)t0 * a.y_stride + row0 + (at & 15);
    auto each = [&](auto&& f) {
      float* y = y0;
#pragma unroll
      for (int j = 0; j < JT; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (t0 + 16 * j + i < a.tokens) {
#pragma unroll
            for (int r = 0; r < RT; ++r)
              if (16 * r < left) f(y[16 * r], r, j, i);
          }
          y += a.y_stride;
        }
        y += 12 * a.y_stride;
      }
    };
    if (add) {
      floatx4 was[RT][JT];
      each([&](float& v, int r, int j, int i) { was[r][j][i] = v; });
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < JT; ++j) tot[r][j] += was[r][j];
    }
    each([&](float& v, int r, int j, int i) { v = tot[r][j][i]; });
  };
  // One group's totals go out to y every 8 chunks, where the next ones are added
  // to them, and start again: each add to them rounds in proportion to what they have reached (16 chunks of Q4_K in one
  // run: 1.24e-7 against 64 bits, an fp32 evaluation 1.17e-7)
  constexpr int kSegment = 8;

  const int iters = (a.chunks + KW - 1) / KW;
  bool large = false;  // 32-block types: a large scale among this lane's
  if (kw < a.chunks) {
    load_rows(kw);
    load_x(kw);
    split_x(lds);
  }
  __syncthreads();
  for (int it = 0; it < iters; ++it) {
    const int c = it * KW + kw;
    uint8_t* buf = lds + (it & 1) * L::kBytes;
    if (c < a.chunks) {
      const bool more = c + KW < a.chunks;
      if (more) load_x(c + KW);
      __builtin_amdgcn_sched_barrier(0);
      typename W::Scale sc[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        W::prepare(sc[r], raw[r], g);
        if constexpr (W::kBlocks32) large |= sc[r].large;
      }
      // the small products have sums of their own where registers allow: each
      // add rounds in proportion to the sum it meets
      constexpr bool kOwnLo = RT * JT <= 8;
      floatx4 blk[RT][JT], low[kOwnLo ? RT : 1][kOwnLo ? JT : 1];
      floatx4 half[W::kMin ? RT : 1][W::kMin ? JT : 1];  // Q4_K: the first steps' hi products
      const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
      // operand i = (step i / JT, token tile i % JT), read one ahead
      const uint32_t unit = opaque((uint32_t)lane);
      auto operand = [&](int i, half8v& hi, half8v& lo) {
        const int st = i / JT;
        const uint8_t* at = buf + 16 * (unit ^ (uint32_t)st) + (i % JT) * 16384 + st * 2048;
        hi = *reinterpret_cast<const half8v*>(at);
        lo = *reinterpret_cast<const half8v*>(at + 1024);
      };
      half8v ah[2], al[2], bh[RT], bl[RT];
      operand(0, ah[0], al[0]);
#pragma unroll
      for (int i = 0; i < 8 * JT; ++i) {
        const int st = i / JT, j = i % JT;
        if (j == 0) {
#pragma unroll
          for (int r = 0; r < RT; ++r) W::frag(bh[r], bl[r], raw[r], sc[r], st);
        }
        if (i + 1 < 8 * JT) operand(i + 1, ah[(i + 1) & 1], al[(i + 1) & 1]);
        const half8v h = ah[i & 1], l = al[i & 1];
        auto low_sum = [&](int r) -> floatx4& { return kOwnLo ? low[kOwnLo ? r : 0][kOwnLo ? j : 0] : blk[r][j]; };
#pragma unroll
        for (int r = 0; r < RT; ++r) low_sum(r) = mfma_f16(l, bh[r], st ? low_sum(r) : zero);
        if constexpr (W::kPair)
#pragma unroll
          for (int r = 0; r < RT; ++r) low_sum(r) = mfma_f16(h, bl[r], low_sum(r));
        if constexpr (W::kMin)
          if (st == 4)
#pragma unroll
            for (int r = 0; r < RT; ++r) half[r][j] = blk[r][j];
#pragma unroll
        for (int r = 0; r < RT; ++r)
          blk[r][j] = mfma_f16(h, bh[r], (kOwnLo && st == 0) || (W::kMin && st == 4) ? zero : blk[r][j]);
        if (j == JT - 1) __builtin_amdgcn_sched_barrier(0);
      }
      typename W::Finish fin[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) W::finish(fin[r], raw[r], sc[r], g);
      if (more) load_rows(c + KW);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        const floatx4 inv = *reinterpret_cast<const floatx4*>(buf + L::kInv + 64 * j + 16 * g);
        u32x4 sums = {0u, 0u, 0u, 0u};
        if constexpr (W::kMin) {
          sums = *reinterpret_cast<const u32x4*>(buf + L::kSums + j * 1024 + 16 * lane);
          sums[3] = 0u;  // never written
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          if constexpr (kOwnLo) blk[r][j] += low[r][j];
          if constexpr (W::kMin) blk[r][j] += half[r][j];
          add_products<W>(tot[r][j], blk[r][j], inv, fin[r], sums);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) split_x(lds + ((it + 1) & 1) * L::kBytes);
      if (KW == 1 && more && it % kSegment == kSegment - 1) {
        store_rows(it >= kSegment);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int j = 0; j < JT; ++j) tot[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
    __syncthreads();
  }

  bool anew = false;
  if constexpr (W::kBlocks32) {
    anew = __any(large);
    if (anew) [[unlikely]]
      sum_in_parts<W, RT, JT>(tot, a, wbase, woff, tok0, kw, KW, lane);
  }
  if constexpr (KW > 1) {
    floatx4* red = reinterpret_cast<floatx4*>(smem);  // [KW - 1][RW][RT * JT][64]
    if (kw > 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < JT; ++j)
          red[(((kw - 1) * RW + rw) * RT * JT + r * JT + j) * 64 + lane] = tot[r][j];
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int q = 0; q < KW - 1; ++q)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < JT; ++j)
          tot[r][j] += red[((q * RW + rw) * RT * JT + r * JT + j) * 64 + lane];
  }
  store_rows(iters > kSegment && KW == 1 && !anew);
}

// ---------------------------------------------------------------- F32 rows
// Tiles of 32 rows x 16 JT tokens on v_mfma_f32_16x16x4_f32; the workgroup's
// eight waves deal the 16-element pieces of K among themselves (lane (n, g)
// loads elements 4g .. 4g + 3 of a piece of row or token n: 64 contiguous
// bytes a row).  Each token's sums run in one
// order whatever the batch and JT.  Bound by the loads' latency at few tokens
// (512 x 2048, 7 tokens: 19.8 -> 11.7 us), by the fp32 MFMA at many (2048 x
// 4096, 512 tokens: 3.6 ms in passes of four tokens on the VALU -> 0.12 to
// 0.14 ms, 63 to 70 of 157 TFLOP/s); errors against 64 bits 0.8e-7 to 1.0e-7 (0.8e-7 to
// 1.6e-7 before).
constexpr int kF32Waves = 8;
template <int JT>
__global__ void __launch_bounds__(64 * kF32Waves)
gemm_f32_kernel(GemmArgs a) {
  constexpr int RT = 2, PIECES = 4;  // pieces in flight per wave
  __shared__ floatx4 red[kF32Waves - 1][RT * JT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16 * RT, tok0 = blockIdx.y * 16 * JT;
  const float* wr[RT];
  const float* xr[JT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    wr[r] = reinterpret_cast<const float*>(a.w) + (int64_t)min(row0 + 16 * r + n, a.rows - 1) * a.K + 4 * g;
#pragma unroll
  for (int j = 0; j < JT; ++j)
    xr[j] = a.x + (int64_t)min(tok0 + 16 * j + n, a.tokens - 1) * a.x_stride + 4 * g;
  floatx4 tot[RT][JT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < JT; ++j) tot[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 16 * PIECES * wave; k0 < a.K; k0 += 16 * PIECES * kF32Waves) {
    floatx4 w[PIECES][RT], x[PIECES][JT];
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      const int k = k0 + 16 * p;
      const bool in = k + 4 * g < a.K;  // K is a multiple of 4
#pragma unroll
      for (int r = 0; r < RT; ++r)
        w[p][r] = in ? (floatx4)*reinterpret_cast<const floatx4a4*>(wr[r] + k) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < JT; ++j)
        x[p][j] = in ? (floatx4)*reinterpret_cast<const floatx4a4*>(xr[j] + k) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
    // every product in a sum of its own (four elements), added pairwise: a
    // piece's four products in one running sum were 20% further off 64 bits
    // than the VALU's sums had been at K = 424
    floatx4 sum[PIECES][RT][JT];
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < JT; ++j) {
          const floatx4 &u = x[p][j], &v = w[p][r];
          sum[p][r][j] = (mfma4f32(u[0], v[0], zero) + mfma4f32(u[1], v[1], zero)) +
                         (mfma4f32(u[2], v[2], zero) + mfma4f32(u[3], v[3], zero));
        }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int j = 0; j < JT; ++j)
        tot[r][j] += (sum[0][r][j] + sum[1][r][j]) + (sum[2][r][j] + sum[3][r][j]);
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < RT * JT; ++i) red[wave - 1][i][lane] = tot[i / JT][i % JT];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < RT * JT; ++i) {
    floatx4& t = tot[i / JT][i % JT];
    static_assert(kF32Waves == 8, "the sum below");
    t = ((t + red[0][i][lane]) + (red[1][i][lane] + red[2][i][lane])) +
        ((red[3][i][lane] + red[4][i][lane]) + (red[5][i][lane] + red[6][i][lane]));
    const int row = row0 + 16 * (i / JT) + n;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int tok = tok0 + 16 * (i % JT) + 4 * g + e;
      if (row < a.rows && tok < a.tokens) a.y[(int64_t)tok * a.y_stride + row] = t[e];
    }
  }
}

// F32 rows of two to four tokens: a workgroup takes 8 / NT rows and its
// waves take turns at the columns, a float4 of each row and token per lane
// and turn, straight from memory.  Bound by latency up to some thousand rows:
// a wave's loads of one turn are all in flight together, and nothing is
// staged.  Against rows read from LDS-staged tokens by one wave each, and
// against the MFMA tiles below five tokens: 512 x 2048, 2 tokens 6.5 and 10.8
// -> 3.9 us; 1024 x 4096, 4 tokens 28.0 and 20.4 -> 6.2 us; 20000 x 2048, 2
// tokens 36.5 and 46.0 -> 28.6 us (5.7 TB/s).  From five tokens on the tiles
// win: 512 x 2048, 5 tokens 15.0 -> 11.2 us.
constexpr int kFewWaves = 4, kFewSums = 8;
template <int NT>
__global__ void __launch_bounds__(64 * kFewWaves)
gemm_f32_few_kernel(GemmArgs a) {
  constexpr int R = kFewSums / NT;
  __shared__ float red[kFewWaves][kFewSums];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * R;
  const float* wr[R];
  const float* xr[NT];
#pragma unroll
  for (int r = 0; r < R; ++r)
    wr[r] = reinterpret_cast<const float*>(a.w) + (int64_t)min(row0 + r, a.rows - 1) * a.K;
#pragma unroll
  for (int t = 0; t < NT; ++t) xr[t] = a.x + (int64_t)min(t, a.tokens - 1) * a.x_stride;
  float acc[R][NT] = {};
#pragma unroll 2
  for (int k = 4 * (64 * wave + lane); k < a.K; k += 4 * 64 * kFewWaves) {  // K is a multiple of 4
    floatx4 w[R], x[NT];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = *reinterpret_cast<const floatx4a4*>(wr[r] + k);
#pragma unroll
    for (int t = 0; t < NT; ++t) x[t] = *reinterpret_cast<const floatx4a4*>(xr[t] + k);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[r][t] += fmaf(w[r][1], x[t][1], w[r][0] * x[t][0]) + fmaf(w[r][3], x[t][3], w[r][2] * x[t][2]);
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float v = segment_sum<kWave>(acc[r][t]);
      if (lane == 0) red[wave][r * NT + t] = v;
    }
  __syncthreads();
  if (threadIdx.x >= kFewSums) return;
  const int row = row0 + threadIdx.x / NT, t = threadIdx.x % NT;
  if (row < a.rows && t < a.tokens)
    a.y[(int64_t)t * a.y_stride + row] = (red[0][threadIdx.x] + red[1][threadIdx.x]) +
                                         (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

// ------------------------------------------------------------------ host
static hipError_t launch_f32(const GemmArgs& a, bool one_order, hipStream_t stream) {
  if (a.tokens <= 4 && !one_order) {
    const auto kernel = a.tokens <= 2 ? gemm_f32_few_kernel<2> : gemm_f32_few_kernel<4>;
    const int rows = kFewSums / (a.tokens <= 2 ? 2 : 4);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.rows + rows - 1) / rows)),
                       dim3(64 * kFewWaves), 0, stream, a);
    return hipGetLastError();
  }
  const unsigned rows = (unsigned)((a.rows + 31) / 32);
  if (a.tokens <= 16)
    hipLaunchKernelGGL(gemm_f32_kernel<1>, dim3(rows), dim3(64 * kF32Waves), 0, stream, a);
  else
    hipLaunchKernelGGL(gemm_f32_kernel<2>, dim3(rows, (a.tokens + 31) / 32), dim3(64 * kF32Waves), 0,
                       stream, a);
  return hipGetLastError();
}

template <int TYPE, int RT, int KW>
static hipError_t launch_few(const GemmArgs& a, hipStream_t stream) {
  const dim3 grid((a.rows + 16 * RT - 1) / (16 * RT), (a.tokens + 15) / 16);
  hipLaunchKernelGGL((gemm_few_kernel<TYPE, RT, KW>), grid, dim3(64 * KW), 0, stream, a);
  return hipGetLastError();
}

template <int TYPE, int RT, int JT, int RW, int KW>
static hipError_t launch_many(const GemmArgs& a_in, hipStream_t stream) {
  GemmArgs a = a_in;
  a.row_tiles = (a.rows + 16 * RT * RW - 1) / (16 * RT * RW);
  a.token_tiles = (a.tokens + 16 * JT - 1) / (16 * JT);
  const int total = a.row_tiles * a.token_tiles;
  constexpr int lds = KW * 2 * GemmLds<TYPE, JT>::kBytes;
  static_assert(lds <= (int)kMaxLdsBytes && (KW - 1) * RW * RT * JT * 1024 <= lds, "LDS");
  const auto kernel = gemm_many_kernel<TYPE, RT, JT, RW, KW>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(64 * RW * KW), lds,
                     stream, a);
  return hipGetLastError();
}

template <int TYPE>
static hipError_t launch_type(const GemmArgs& a, bool one_order, hipStream_t stream) {
  // one shape for every batch: the one in the middle (64 x 16)
  if (one_order) return launch_many<TYPE, 2, 1, 2, 4>(a, stream);
  // The tile shape whose workgroups, one to a CU, finish first: rounds of
  // workgroups times a workgroup's time, in 0.1 us for 16 chunks of Q4_K
  // (measured with one round).  Small tiles leave fewer CUs idle, large ones
  // decode and split less per product: 256 x 64 does 172 rows x tokens a us,
  // 128 x 32 117, 32 x 16 40.  With other chunk counts and types only the
  // proportions matter: of 70 calls (Q4_K of 2, 16 and 56 chunks, Q6_K of 16
  // and 56, Q8_0 of 11, Q5_0 of 4; 1024 to 14336 rows, 4 to 500 tokens) the
  // shape taken was within 3% of the fastest of the eight in 63, and 6 to 24%
  // off where rows are short or three token tiles of a pair type meet 64 row
  // tiles (Q4_K 14336 x 512, 7 tokens: 5.6 us, 4.5 in 64 x 16 tiles of many).
  struct Shape {
    int rows, tokens, base, per_token;  // per_token: of the first 16 tokens
  };
  static constexpr Shape shapes[] = {
      {64, 16, 138, 3}, {32, 16, 95, 3}, {16, 16, 77, 2},             // few
      {32, 16, 128, 0}, {64, 16, 166, 0}, {128, 32, 350, 0},          // many
      {128, 64, 670, 0}, {256, 64, 950, 0}};
  const int64_t cus = device_cu_count();
  int best = 0;
  int64_t least = INT64_MAX;
  for (int i = 0; i < (int)(sizeof shapes / sizeof shapes[0]); ++i) {
    const Shape& s = shapes[i];
    const int64_t groups = (int64_t)((a.rows + s.rows - 1) / s.rows) * ((a.tokens + s.tokens - 1) / s.tokens);
    const int64_t time = (groups + cus - 1) / cus * (s.base + s.per_token * std::min(a.tokens, 16));
    if (time < least) {
      least = time;
      best = i;
    }
  }
  switch (best) {
    case 0: return launch_few<TYPE, 4, 8>(a, stream);
    case 1: return launch_few<TYPE, 2, 8>(a, stream);
    case 2: return launch_few<TYPE, 1, 8>(a, stream);
    case 3: return launch_many<TYPE, 1, 1, 2, 4>(a, stream);
    case 4: return launch_many<TYPE, 2, 1, 2, 4>(a, stream);
    case 5: return launch_many<TYPE, 2, 2, 4, 2>(a, stream);
    case 6: return launch_many<TYPE, 1, 4, 8, 1>(a, stream);
    default: return launch_many<TYPE, 2, 4, 8, 1>(a, stream);
  }
}

static hipError_t launch(int type, const GemmArgs& a, bool one_order, hipStream_t stream) {
  switch (type) {
    case kQ4_K: return launch_type<kQ4_K>(a, one_order, stream);
    case kQ6_K: return launch_type<kQ6_K>(a, one_order, stream);
    case kQ5_0: return launch_type<kQ5_0>(a, one_order, stream);
    case kQ8_0: return launch_type<kQ8_0>(a, one_order, stream);
    case kF32: return launch_f32(a, one_order, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t gemm_launch(const GemvProblem& p, hipStream_t stream) {
  if (p.tokens < 1 || p.rows < 1 || p.rows > INT32_MAX || p.columns % block_weights(p.type))
    return hipErrorInvalidValue;
  // 16-byte loads of Q4_K rows, 4-byte floats, dword loads at or below the
  // other types'; F32 rows of whole float4s
  if (reinterpret_cast<uintptr_t>(p.weights) % (p.type == kQ4_K ? 16 : p.type == kF32 ? 4 : 2))
    return hipErrorInvalidValue;
  if (p.type == kF32 && p.columns % 4) return hipErrorInvalidValue;
  // lane offsets within a tile are 32 bits
  if (p.x_stride < 0 || p.x_stride > (1 << 22) || p.row_bytes > (1 << 22)) return hipErrorInvalidValue;
  // A grid has less than 2^32 threads and at most 65535 workgroups in its
  // second dimension: launches of at most 2^20 rows and as many tokens as
  // 2^22 tiles of 16 x 16, the smallest, hold (whole tiles of every shape)
  const int64_t row_span = std::min<int64_t>(p.rows, 1 << 20), row_tiles = (row_span + 15) / 16;
  const int64_t token_span = 64 * (std::min<int64_t>(65535, (1 << 22) / row_tiles) / 4);
  for (int64_t r0 = 0; r0 < p.rows; r0 += row_span)
    for (int64_t t0 = 0; t0 < p.tokens; t0 += token_span) {
      GemmArgs a{};
      a.w = p.weights + r0 * p.row_bytes;
      a.row_bytes = p.row_bytes;
      a.rows = (int)std::min(row_span, p.rows - r0);
      a.K = (int)p.columns;
      a.chunks = (a.K + 255) / 256;
      a.x = p.x + t0 * p.x_stride;
      a.x_stride = p.x_stride;
      a.tokens = (int)std::min(token_span, p.tokens - t0);
      a.y = p.y + t0 * p.y_stride + r0;
      a.y_stride = p.y_stride;
      const hipError_t e = launch(p.type, a, p.one_order, stream);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

}  // namespace llhip
