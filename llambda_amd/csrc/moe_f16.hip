// moe_f16.hip -- grouped expert products of K-quant swiglu layers (Qwen3Next:
// Q4_K / Q6_K slabs in the tile-major layout, hidden and ffn widths of whole
// 256-element chunks), batches of two or more tokens.
//
// The operands are those of gemm_f16.h: activations as f16 hi + lo with one
// power-of-two scale per (token, 256-element chunk), codes as exact f16
// integers or pairs, so a chunk's sums need no scaling per group and the VALU
// only unpacks codes.  Activations are kept as operand images: row r of K
// elements holds, per chunk, 512 bytes of hi and 512 of lo parts, 16 bytes per
// (step, lane group), so an MFMA operand is one 16-byte load per lane; beside
// them, per (chunk, lane group), 16 bytes: the Q4_K sums' operand (12 bytes)
// and the fp32 1 / scale.  x's images are formed once per layer, in memory;
// the activations silu(g) * u leave the up products as fp32 rows, and each
// workgroup of the down products forms their images in LDS (a chunk's scale
// needs all 256 values, which several workgroups produce).
//
// Every output's sums run in one order whatever the batch: chunk after chunk,
// step after step, lo before hi.
#include "activations.h"
#include "moe.h"
#include "moe_f16.h"

#include <algorithm>

namespace llhip {

constexpr int kWaves = 8;  // per workgroup: two workgroups per CU
// Chunks of the down products' K held in LDS: two (ffn 512, the Qwen3Next
// layers') leave two workgroups to a CU at two token tiles (70 KB).  Four would
// fit (139 KB, one workgroup); wider ffn keep the bf16 pipelines, unmeasured
// here.
constexpr int kDownChunks = 2;

// ------------------------------------------------------------- products
// Activations reach the products through LDS: one operand (a step's hi or lo
// part of 16 tokens) is 1 KB, each lane's 16 bytes fetched by DMA from its
// token's row, so every wave of the workgroup reads what one of them staged.
// A chunk's image: [token tile][step][hi, lo][lane].  Where the workgroup forms
// the image itself, lane l's 16 bytes of a step sit at position l ^ step, which
// spreads the quads of a row over the banks (SWIZZLE).
constexpr int kTileImage = 16384;

// 16 bytes per lane from each lane's address to LDS image + 16 * lane.
__device__ __forceinline__ void dma16(const uint8_t* from, uint8_t* image) {
  const uint32_t at = __builtin_amdgcn_readfirstlane(lds_address(image));
  asm volatile(
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off"
      :
      : "v"(from), "{m0}"(at)
      : "memory");
}

// The waves of a workgroup stage chunk images: xp[j] = this lane's token row's
// chunk, offset to its lane group.
template <int JT>
__device__ __forceinline__ void stage_chunk(const uint8_t* const (&xp)[JT], uint8_t* image, int wave) {
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int o = 0; o < 16 / kWaves; ++o) {
      const int op = wave * (16 / kWaves) + o;  // step op >> 1, lo for odd op
      dma16(xp[j] + 64 * (op >> 1) + 512 * (op & 1), image + j * kTileImage + 1024 * op);
    }
}

// One chunk of two row tiles against JT token tiles: tot += W x.
template <typename W, int JT, bool SWIZZLE>
__device__ __forceinline__ void expert_chunk(floatx4 (&tot)[2][JT], const typename W::Raw (&raw)[2],
                                             const uint8_t* image, u32x4 (&side)[JT], int lane) {
  const int g = lane >> 4;
  floatx4 blk[2][JT];
  typename W::Scale sc[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) W::prepare(sc[r], raw[r], g);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    half8v bh[2], bl[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) W::frag(bh[r], bl[r], raw[r], sc[r], s);
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const uint8_t* at = image + j * kTileImage + 2048 * s + 16 * (SWIZZLE ? lane ^ s : lane);
      const half8v ah = *reinterpret_cast<const half8v*>(at);
      const half8v al = *reinterpret_cast<const half8v*>(at + 1024);
#pragma unroll
      for (int r = 0; r < 2; ++r)
        blk[r][j] = mfma_f16(al, bh[r], s ? blk[r][j] : floatx4{0.f, 0.f, 0.f, 0.f});
      if constexpr (W::kPair)
#pragma unroll
        for (int r = 0; r < 2; ++r) blk[r][j] = mfma_f16(ah, bl[r], blk[r][j]);
#pragma unroll
      for (int r = 0; r < 2; ++r) blk[r][j] = mfma_f16(ah, bh[r], blk[r][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    const uint32_t bits = side[j][3];  // (a bit_cast of the element itself reads element 0)
    const float own = __builtin_bit_cast(float, bits);
    floatx4 inv;
#pragma unroll
    for (int i = 0; i < 4; ++i) inv[i] = __shfl(own, 4 * g + i);
    side[j][3] = 0u;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      typename W::Finish fin;
      W::finish(fin, raw[r], sc[r], g);
      add_products<W>(tot[r][j], blk[r][j], inv, fin, side[j]);
    }
  }
}

// The chunk table entry and row group of this workgroup: false past the table.
// A 1-D grid in which the `groups` row groups of entry c take the workgroups
// (c / 8) * 8 groups + 8 k + c % 8: workgroups are dealt to the eight XCDs by
// id modulo 8, so an entry's row groups run on one XCD, close in time, and its
// activations are fetched into that L2 once.
struct ExpertEntry {
  MoeChunk chunk;
  bool shared;
  int group;
};
__device__ __forceinline__ bool expert_entry(const MoeGemmArgs& a, ExpertEntry& e) {
  const int groups = a.row_tiles, id = blockIdx.x;
  const int i = id / (8 * groups) * 8 + (id & 7);
  const int c0 = a.chunk_counts[0], c1 = a.joint ? a.chunk_counts[1] : 0;
  if (i >= c0 + c1) return false;
  e.chunk = a.chunks[i];
  e.shared = i >= c0;
  e.group = (id >> 3) % groups;
  return true;
}
// The pair at position p of the entry (past its last: the last).
__device__ __forceinline__ int entry_pair(const MoeGemmArgs& a, const MoeChunk& c, int p) {
  return a.perm[c.start + min(p, c.count - 1)];
}

// Gate and up rows and silu(g) * u: a workgroup takes one entry's 16 JT pairs
// and 128 ffn rows, wave w gate and up rows 16 w .. 16 w + 15 over all of K.  A
// chunk's rows (registers) and activations (LDS, two images in turn, one
// barrier per chunk) are requested while the chunk before is multiplied; the
// two workgroups of a CU cover each other's starts, waits and ends.
// DEEP, for grids of at most one workgroup per CU, whose waves have no other
// to wait behind: all of K's activations are staged at the start, and each
// wave keeps the rows of the next three chunks in flight (the same sums in the
// same order; 2 tokens of a Qwen3Next layer: 63 -> 47 us with the down launch's
// shorter workgroups; from 344 workgroups on the two that share a CU win: 8
// tokens 83 us deep, 76 not, 256 tokens 352 and 315).
// Measured for 256 tokens (E 512, top 10, 634 MB of rows): 153 to 163 us, 4.0
// TB/s (177 us with bf16 parts, whose group sums the VALU scaled; 180 us as one
// workgroup of 16 waves per CU, whose start, end and waits nothing covered).
// The VALU issues for 53% of the SIMD cycles (9.4 instructions per MFMA: most
// experts have 5 pairs of the tile's 16) and the matrix cores work for 23.
template <int TYPE, int JT, bool DEEP>
__global__ void __launch_bounds__(64 * kWaves, JT == 1 && !DEEP ? 4 : 2)
expert_up_kernel(MoeGemmArgs a) {
  using W = ExpertW<TYPE>;
  extern __shared__ __align__(16) uint8_t images[];  // [DEEP ? chunks : 2][JT * kTileImage]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = lane & 15, g = lane >> 4;
  ExpertEntry e;
  if (!expert_entry(a, e)) return;
  const int rows = e.shared ? a.s_N : a.N, f0 = (e.group * kWaves + wave) * 16;
  if (e.group * kWaves * 16 >= rows) return;
  const int chunks = a.K >> 8;
  const int64_t slab = e.shared ? 0 : e.chunk.expert * a.expert_stride;
  const int64_t tile = (int64_t)(f0 >> 4) * chunks * 16 * W::kPitch;
  const uint8_t* w0 = (e.shared ? a.s_w0 : a.w0) + slab + tile;
  const uint8_t* w1 = (e.shared ? a.s_w1 : a.w1) + slab + tile;
  const uint32_t own = (uint32_t)n * W::kPitch;
  auto load_rows = [&](typename W::Raw(&raw)[2], int c) {
    const uint32_t at = (uint32_t)c * 16 * W::kPitch;
    W::load(raw[0], w0 + at, own, g, 8);
    W::load(raw[1], w1 + at, own, g, 8);
  };
  constexpr int AHEAD = DEEP ? 3 : 1;  // chunks of rows in flight
  typename W::Raw raw[AHEAD + 1][2];
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) load_rows(raw[d], min(d, chunks - 1));
  const uint8_t* xp[JT];
  const u32x4* sp[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    const int q = entry_pair(a, e.chunk, 16 * j + n);
    const int t = q >= a.pairs ? q - a.pairs : q / a.top_k;
    xp[j] = reinterpret_cast<const uint8_t*>(a.aq + t * a.aq_stride) + 16 * g;
    sp[j] = reinterpret_cast<const u32x4*>(a.as + t * a.as_stride) + g;
  }
  for (int c = 0; c < (DEEP ? chunks : 1); ++c) {
    stage_chunk<JT>(xp, images + c * JT * kTileImage, wave);
#pragma unroll
    for (int j = 0; j < JT; ++j) xp[j] += 1024;
  }
  u32x4 side[AHEAD + 1][JT];
#pragma unroll
  for (int d = 0; d < AHEAD; ++d)
#pragma unroll
    for (int j = 0; j < JT; ++j) side[d][j] = sp[j][4 * min(d, chunks - 1)];
  floatx4 tot[2][JT];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int j = 0; j < JT; ++j) tot[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (DEEP) {
    wait_loads<0>();  // this wave's part of the images
    __syncthreads();
  }
  for (int c0 = 0; c0 < chunks; c0 += AHEAD + 1) {
#pragma unroll
    for (int d = 0; d <= AHEAD; ++d) {
      const int c = c0 + d;
      if (c < chunks) {
        if constexpr (!DEEP) {
          wait_loads<0>();  // this wave's part of image c, and its rows
          __syncthreads();
        }
        constexpr int N = AHEAD + 1;
        const int ahead = min(c + AHEAD, chunks - 1), slot = (d + AHEAD) % N;
        load_rows(raw[slot], ahead);
#pragma unroll
        for (int j = 0; j < JT; ++j) side[slot][j] = sp[j][4 * ahead];
        if (!DEEP && c + 1 < chunks) {
          stage_chunk<JT>(xp, images + ((c + 1) & 1) * JT * kTileImage, wave);
#pragma unroll
          for (int j = 0; j < JT; ++j) xp[j] += 1024;
        }
        expert_chunk<W, JT, false>(tot, raw[d], images + (DEEP ? c : c & 1) * JT * kTileImage,
                                   side[d], lane);
      }
    }
  }
  // ffn row f0 + n, pair 16 j + 4 g + i
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma clang fp contract(off)
      const float h = silu_ref(tot[0][j][i]) * tot[1][j][i];  // llambda.lisp:5386-5401
      const int p = 16 * j + 4 * g + i;
      if (p < e.chunk.count)
        reinterpret_cast<float*>(a.oq + entry_pair(a, e.chunk, p) * a.oq_stride)[f0 + n] = h;
    }
}

// Down rows, fp32 outputs per pair: a workgroup forms its entry's images once
// (K of at most kDownChunks chunks), then its waves take two row tiles at a
// time over all of K, the rows of the next step always in flight.  256 tokens
// as above (457 MB of rows): 125 to 132 us (174 us with bf16 parts in 16-wide
// products); VALU 51% of the SIMD cycles, matrix cores 19.
template <int TYPE, int JT>
__global__ void __launch_bounds__(64 * kWaves, JT == 1 ? 4 : 2)
expert_down_kernel(MoeGemmArgs a) {
  using W = ExpertW<TYPE>;
  // [chunks][JT * kTileImage], then the side entries [chunks][JT][64 lanes]
  extern __shared__ __align__(16) uint8_t images[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = lane & 15, g = lane >> 4;
  ExpertEntry e;
  if (!expert_entry(a, e)) return;
  const int rows = e.shared ? a.s_N : a.N, chunks = (e.shared ? a.s_K : a.K) >> 8;
  const int tiles = rows >> 4, step = 2 * kWaves * a.row_tiles;
  int tile = 2 * (kWaves * e.group + wave);
  const uint8_t* w = e.shared ? a.s_w0 : a.w0 + e.chunk.expert * a.expert_stride;
  const uint32_t tile_bytes = (uint32_t)chunks * 16 * W::kPitch, own = (uint32_t)n * W::kPitch;
  auto load_rows = [&](typename W::Raw(&raw)[2], int t, int c) {
    const uint8_t* b = w + (int64_t)min(t, tiles - 2) * tile_bytes + (uint32_t)c * 16 * W::kPitch;
    W::load(raw[0], b, own, g, 8);
    W::load(raw[1], b + tile_bytes, own, g, 8);
  };
  typename W::Raw raw[2];
  load_rows(raw, tile, 0);
  u32x4* sides = reinterpret_cast<u32x4*>(images + chunks * JT * kTileImage);
  for (int i = wave; i < 16 * JT * chunks; i += kWaves) {
    const int c = i / (16 * JT), p = i - c * 16 * JT;  // pairs past the count: the last's
    const float* row = reinterpret_cast<const float*>(a.aq + entry_pair(a, e.chunk, p) * a.aq_stride);
    const floatx4 v = *reinterpret_cast<const floatx4*>(row + 256 * c + 4 * lane);
    uint2 hi, lo;
    u32x4 side;
    split_chunk<W>(v, lane, hi, lo, side);
    int pg, ps, high;
    W::place(lane, pg, ps, high);
    const int j = p >> 4, t = p & 15;
    uint8_t* at = images + (c * JT + j) * kTileImage + 2048 * ps + 16 * ((t + 16 * pg) ^ ps) + 8 * high;
    *reinterpret_cast<uint2*>(at) = hi;
    *reinterpret_cast<uint2*>(at + 1024) = lo;
    if ((lane & 15) == 0) sides[(c * JT + j) * 64 + t + lane] = side;  // lane = 16 group
  }
  float* out[JT][4];  // pairs 16 j + 4 g + i
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[j][i] = a.out + entry_pair(a, e.chunk, 16 * j + 4 * g + i) * a.out_stride + n;
  __syncthreads();
  for (; tile < tiles; tile += step) {
    floatx4 tot[2][JT];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int j = 0; j < JT; ++j) tot[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < chunks; ++c) {
      typename W::Raw next[2];
      u32x4 side[JT];
      const bool more = c + 1 < chunks;
      load_rows(next, more ? tile : tile + step, more ? c + 1 : 0);
#pragma unroll
      for (int j = 0; j < JT; ++j) side[j] = sides[(c * JT + j) * 64 + lane];
      expert_chunk<W, JT, true>(tot, raw, images + c * JT * kTileImage, side, lane);
#pragma unroll
      for (int r = 0; r < 2; ++r) raw[r] = next[r];
    }
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * j + 4 * g + i < e.chunk.count)
#pragma unroll
          for (int r = 0; r < 2; ++r) out[j][i][16 * (tile + r)] = tot[r][j][i];
  }
}

// ------------------------------------------------------------------ host
bool moe_f16_supported(const MoePlan& p) {
  auto k = [](int type) { return type == kQ4_K || type == kQ6_K; };
  return p.variant == kQwen3Next && k(p.up_type) && p.gate_type == p.up_type && k(p.down_type) &&
         p.hidden % 256 == 0 && p.ffn % 256 == 0 && p.ffn <= 256 * kDownChunks &&
         (p.shared_ffn == 0 || (p.sh_up_type == p.up_type && p.sh_gate_type == p.up_type &&
                                p.sh_down_type == p.down_type && p.shared_ffn % 256 == 0 &&
                                p.shared_ffn <= 256 * kDownChunks));
}

static hipError_t launch_lds(void (*kernel)(MoeGemmArgs), dim3 grid, dim3 block, int lds,
                             hipStream_t stream, const MoeGemmArgs& a) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, a);
  return hipGetLastError();
}

hipError_t moe_f16_up_launch(int type, const MoeGemmArgs& a_in, int token_tiles, int max_chunks,
                             hipStream_t stream) {
  MoeGemmArgs a = a_in;
  a.row_tiles = std::max(a.N, a.joint ? a.s_N : 0) / (16 * kWaves);
  const dim3 grid((max_chunks + 7) / 8 * 8 * a.row_tiles), block(64 * kWaves);
  const bool deep = (int)grid.x <= device_cu_count() && token_tiles == 1 && a.K <= 2048;
  const int lds = (deep ? a.K / 256 : 2) * token_tiles * kTileImage;
  void (*kernel)(MoeGemmArgs) = nullptr;
  if (type == kQ4_K)
    kernel = deep               ? expert_up_kernel<kQ4_K, 1, true>
             : token_tiles == 1 ? expert_up_kernel<kQ4_K, 1, false>
                                : expert_up_kernel<kQ4_K, 2, false>;
  else if (type == kQ6_K)
    kernel = deep               ? expert_up_kernel<kQ6_K, 1, true>
             : token_tiles == 1 ? expert_up_kernel<kQ6_K, 1, false>
                                : expert_up_kernel<kQ6_K, 2, false>;
  else
    return hipErrorInvalidValue;
  return launch_lds(kernel, grid, block, lds, stream, a);
}

hipError_t moe_f16_down_launch(int type, const MoeGemmArgs& a_in, int token_tiles, int max_chunks,
                               hipStream_t stream) {
  // row groups of 256 a workgroup's waves share: four per workgroup, one while
  // the launch is short (2 and 8 tokens of a Qwen3Next layer: the layer 49 ->
  // 47 and 76 -> 75 us; 12 tokens, with one group each: 79 -> 85 us)
  MoeGemmArgs a = a_in;
  const int groups = a.N / (32 * kWaves);
  a.row_tiles = max_chunks * groups <= 3 * device_cu_count() ? groups : (groups + 3) / 4;
  const dim3 grid((max_chunks + 7) / 8 * 8 * a.row_tiles), block(64 * kWaves);
  const int lds = (std::max(a.K, a.joint ? a.s_K : 0) / 256) * token_tiles * (kTileImage + 1024);
  void (*kernel)(MoeGemmArgs) = nullptr;
  if (type == kQ4_K)
    kernel = token_tiles == 1 ? expert_down_kernel<kQ4_K, 1> : expert_down_kernel<kQ4_K, 2>;
  else if (type == kQ6_K)
    kernel = token_tiles == 1 ? expert_down_kernel<kQ6_K, 1> : expert_down_kernel<kQ6_K, 2>;
  else
    return hipErrorInvalidValue;
  return launch_lds(kernel, grid, block, lds, stream, a);
}

}  // namespace llhip
