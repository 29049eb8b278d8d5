// moe_f16.h -- expert weights and activation images of the f16 expert products
// (moe_f16.hip) and of the router launch that forms x's images (moe_mfma.hip).
#pragma once

#include "gemm_f16.h"

namespace llhip {

// ------------------------------------------------------------ weights
// Tile-major rows (moe_tile_launch): kPitch bytes apart within a 16-row tile's
// chunk.  place(): the operand slot of quad `i` (elements 4i .. 4i + 3).
template <int TYPE>
struct ExpertW;

// Codes centred (gemm_f16.h).
template <>
struct ExpertW<kQ4_K> : Q4KRow {
  static constexpr int kPitch = 144;
  static constexpr bool kCentred = true;
  struct Scale {
    half2v sl, ol, sh, oh;  // sc / 16 and -72 sc of sub-blocks 2g and 2g + 1
  };
  struct Finish {
    uint32_t m0, m1, m2, c0, c1, c2;  // against the sub-blocks' sums: minima, and 256 sc
    float d, dm;                      // d and -32 dmin
  };
  static __device__ __forceinline__ void place(int i, int& g, int& s, int& high) {
    g = i >> 4;
    s = i & 7;
    high = (i >> 3) & 1;
  }
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int g) {
    const uint32_t sc = scale_bytes(r, g);
    const half2v k1152 = splat2((_Float16)-1152.f);
    c.sl = splat2((_Float16)((float)(sc & 0xFFu) * 0.0625f));
    c.sh = splat2((_Float16)((float)((sc >> 8) & 0xFFu) * 0.0625f));
    c.ol = c.sl * k1152;
    c.oh = c.sh * k1152;
  }
  static __device__ __forceinline__ void finish(Finish& f, const Raw& r, const Scale& c, int g) {
    minima(min_bytes(r, g), f.m0, f.m1, f.m2);
    // (8 sc S = 256 sc S / 32)
    const half2v k4096 = splat2((_Float16)4096.f);
    const half2v c0 = c.sl * k4096, c1 = c.sh * k4096;
    f.c0 = __builtin_bit_cast(uint32_t, c0);
    f.c1 = __builtin_bit_cast(uint32_t, c1);
    f.c2 = __builtin_bit_cast(uint32_t, half2v{c0.x, c1.x});
    f.d = half_bits_to_float(r.h.x & 0xFFFFu);
    f.dm = -32.f * half_bits_to_float(r.h.x >> 16);
  }
  // sc (q - 8) = (1024 + 16 q) sc / 16 - 72 sc, exact in one fma
  static __device__ __forceinline__ void frag(half8v& hi, half8v&, const Raw& r, const Scale& c,
                                              int s) {
    const uint32_t w = codes(r, s), lo = (w << 4) & 0xF0F0F0F0u, hg = w & 0xF0F0F0F0u;
    hi = join8(__builtin_elementwise_fma(bytes02(lo), c.sl, c.ol),
               __builtin_elementwise_fma(bytes13(lo), c.sl, c.ol),
               __builtin_elementwise_fma(bytes02(hg), c.sh, c.oh),
               __builtin_elementwise_fma(bytes13(hg), c.sh, c.oh));
  }
};

// A row's 32-byte runs of ql and qh hold dword 4s + g of the GGUF run at dword
// 2g + s, so lane group g = 2h + b, taking dwords 4b .. 4b + 3 of half h's
// runs, meets GGUF dwords 2b, 2b + 4, 2b + 1, 2b + 5: both 16-element scale
// groups of each of its four runs k, alternating.  Step 2i + kk takes dword i
// of runs k = kk (low) and kk + 2 (high).
template <>
struct ExpertW<kQ6_K> {
  static constexpr int kPitch = 212;
  static constexpr bool kPair = true, kMin = false;
  struct Raw {
    u32x4 la, lb, qh;
    uint2 s;
    uint32_t d;
  };
  struct Scale {
    half2v sc[8];  // 2^-14 times scale 2k + (dword >> 2)
  };
  struct Finish {
    float d;
  };
  static __device__ __forceinline__ void place(int i, int& g, int& s, int& high) {
    const int h = i >> 5, k = (i >> 3) & 3, o = i & 7;
    g = 2 * h + ((o >> 1) & 1);
    s = 2 * (2 * (o & 1) + (o >> 2)) + (k & 1);
    high = k >> 1;
  }
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* b, uint32_t o, int g, int) {
    const uint32_t h = (uint32_t)g >> 1, e = 16u * ((uint32_t)g & 1u);
    const uint8_t* ql = b + (o + 64 * h + e);
    r.la = *reinterpret_cast<const u32x4a4*>(ql);
    r.lb = *reinterpret_cast<const u32x4a4*>(ql + 32);
    r.qh = *reinterpret_cast<const u32x4a4*>(b + (o + 128 + 32 * h + e));
    const uint32_t* sc = reinterpret_cast<const uint32_t*>(b + (o + 192 + 8 * h));
    r.s = make_uint2(sc[0], sc[1]);
    r.d = *reinterpret_cast<const uint32_t*>(b + (o + 208));
  }
  static __device__ __forceinline__ void prepare(Scale& c, const Raw& r, int) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      c.sc[i] = splat2((_Float16)(
          0x1p-14f * (float)(int)(int8_t)(((i < 4 ? r.s.x : r.s.y) >> (8 * (i & 3))) & 0xFFu)));
  }
  static __device__ __forceinline__ void finish(Finish& f, const Raw& r, const Scale&, int) {
    f.d = 0x1p14f * half_bits_to_float(r.d & 0xFFFFu);
  }
  static __device__ __forceinline__ void frag(half8v& hi, half8v& lo, const Raw& r, const Scale& c,
                                              int st) {
    const int i = st >> 1, kk = st & 1, s = i & 1;
    const uint32_t w = kk ? r.lb[i] : r.la[i], v = r.qh[i];
    const uint32_t cl = (w & 0x0F0F0F0Fu) | (((v >> (2 * kk)) & 0x03030303u) << 4);
    const uint32_t ch = ((w >> 4) & 0x0F0F0F0Fu) | (((v >> (2 * kk + 4)) & 0x03030303u) << 4);
    const half2v off = splat2((_Float16)-1056.f);
    half2v h[4], l[4];
    exact_product(bytes02(cl) + off, c.sc[2 * kk + s], h[0], l[0]);
    exact_product(bytes13(cl) + off, c.sc[2 * kk + s], h[1], l[1]);
    exact_product(bytes02(ch) + off, c.sc[2 * kk + 4 + s], h[2], l[2]);
    exact_product(bytes13(ch) + off, c.sc[2 * kk + 4 + s], h[3], l[3]);
    hi = join8(h[0], h[1], h[2], h[3]);
    lo = join8(l[0], l[1], l[2], l[3]);
  }
};

// --------------------------------------------------------- operand images
// One chunk of a row, elements 4 lane .. 4 lane + 3 in v, by one wavefront: the
// lane's quad as hi and lo parts, and the row's side entry of lane group
// lane >> 4, whole in lanes 0, 16, 32 and 48.
template <typename W>
__device__ __forceinline__ void split_chunk(const floatx4& v, int lane, uint2& hi, uint2& lo,
                                            u32x4& side) {
  const float top = wave_max(abs_max4(0.f, v));
  float scale, inv;
  chunk_scale(top, scale, inv);
  split_quad(v, scale, hi, lo);
  if (infinite(top)) lo = make_uint2(drop_inf(hi.x, lo.x), drop_inf(hi.y, lo.y));
  side = u32x4{0u, 0u, 0u, __builtin_bit_cast(uint32_t, inv)};
  if constexpr (W::kMin) {
    // sub-block lane >> 3: eight lanes' quads
    float h = pair_sum(hi.y, pair_sum(hi.x, 0.f)), l = pair_sum(lo.y, pair_sum(lo.x, 0.f));
    h += dpp<kDppXor1>(h);
    l += dpp<kDppXor1>(l);
    h += dpp<kDppXor2>(h);
    l += dpp<kDppXor2>(l);
    h += dpp<kDppHalfMirror>(h);
    l += dpp<kDppHalfMirror>(l);
    if (fabsf(h) == __builtin_inff()) l = 0.f;
    const float h1 = __shfl_down(h, 8), l1 = __shfl_down(l, 8);
    side[0] = split_sum(h);
    side[1] = split_sum(h1);
    side[2] = (uint32_t)lo_sum(l) | ((uint32_t)lo_sum(l1) << 16);
  }
}

}  // namespace llhip
