// BlockFHT generator kernels at block size 2^15 on the matrix cores: forward
// (signed bf16 output slice) and backward (bfloat16 partial rows of the latent
// gradient, one per workgroup).  The chain itself (layouts, Walsh stages, LDS exchanges, sign
// words) is in bfht_mfma_chain.h.
//
// Reference semantics: latent_weight_lab/block_fht.py:84-109 (forward) and
// csrc/block_fht_ext_cuda.cu:185-223 (backward: the same chain with the sign
// layers in reverse order).
#include "bfht_mfma_chain.h"

namespace lwl {
namespace mfma15 {
namespace {

// Runs the chain and leaves this lane's eight signed output chunks in v (odd
// L: from layout F, or from S1 without kDirect; even L: from S0), times `scale` after
// their rounding; chunk k holds block positions chunk_pos<L, kDirect>(x, k) .. + 7.
template <int L, int kBufs, bool kDirect = L % 2 == 1, class SignLayer>
__device__ __forceinline__ void chain_chunks(const Ctx& x, unsigned char* lds, const u32x4 (&src)[kTiles][2],
                                             SignLayer sign_layer, u32x4 (&v)[8], float scale = 1.0f) {
  f32x16 acc[kTiles];
  uint32_t nw[4];
  if constexpr (kDirect) {
    run_chain<L, true, kBufs>(acc, x, lds, src, sign_layer, nw);
    direct_chunks(acc, x, reinterpret_cast<const uint32_t*>(lds + kBufs * kXBufBytes) + (L - 1) * kWordsPerLayer, v,
                  scale);
  } else {
    run_chain<L, false, kBufs>(acc, x, lds, src, sign_layer, nw);
    out_chunks<L>(acc, nw, x, v);
    if (scale != 1.0f) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = scale_chunk(v[k], scale);
    }
  }
}
template <int L, bool kDirect>
__device__ __forceinline__ int chunk_pos(const Ctx& x, int k) {
  return kDirect ? direct_chunk_pos(x, k) : out_chunk_pos<L>(x, k);
}

// Puts the chunks into `lds` in position order (chunk c at stage_slot(c)) and
// waits for every wave's; returns the staged block.
template <int L, int kBufs, bool kDirect = L % 2 == 1>
__device__ __forceinline__ const u32x4* stage_chunks(const u32x4 (&v)[8], const Ctx& x, unsigned char* lds) {
  // two buffers: the one the last layer did not exchange through is free
  u32x4* stage = reinterpret_cast<u32x4*>(lds + (kBufs == 2 ? (L & 1) * kXBufBytes : 0));
  if (kBufs == 1) __syncthreads();  // every wave has read the last exchange
#pragma unroll
  for (int k = 0; k < 8; ++k) stage[stage_slot(chunk_pos<L, kDirect>(x, k) >> 3)] = v[k];
  __syncthreads();
  return stage;
}

// The staged block's chunks, consecutive threads on consecutive 16 bytes,
// write-through; stores past the resource are dropped.
__device__ __forceinline__ void store_staged(const u32x4* stage, __amdgpu_buffer_rsrc_t out_r) {
  constexpr int kPer = kChunks / kThreads;
  u32x4 v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) v[i] = stage[stage_slot(i * kThreads + (int)threadIdx.x)];
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    __builtin_amdgcn_raw_buffer_store_b128(v[i], out_r, (i * kThreads + (int)threadIdx.x) * 16, 0, kStreamStore);
}

// ---------------------------------------------------------------- forward

// The 16 bytes that start M bf16 elements before chunk b: the last M elements
// of chunk a followed by the first 8 - M of b (bytes 16 - 2M .. 31 - 2M of a:b).
template <int M>
__device__ __forceinline__ u32x4 chunk_shifted(const u32x4& a, const u32x4& b) {
  const uint32_t w[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  constexpr int o = 16 - 2 * M, q = o >> 2, r = o & 3;
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (r == 0) v[i] = w[q + i];
    else v[i] = __builtin_amdgcn_alignbyte(w[q + i + 1], w[q + i], r);
  }
  return v;
}

// Stores block positions [lo, hi) of a staged block to oblk (2-byte aligned,
// M = its element offset from a 16-byte boundary): slot j of the aligned grid
// holds positions 8j - M .. 8j - M + 7, built from staged chunks j - 1 and j.
// Slots inside [lo, hi) take one 16-byte store; the slots at the range's ends,
// shared with other blocks' outputs, get element stores of their positions in
// the range.  Slots j = 0 .. kChunks (the last one only exists for M > 0).
template <int M>
__device__ __forceinline__ void store_range_shifted(const u32x4* stage, __bf16* oblk, int lo, int hi) {
  const auto a_r = rsrc(oblk - M, (uint32_t)((kChunks + 1) * 16));
  uint16_t* o16 = reinterpret_cast<uint16_t*>(oblk);
  constexpr int kPer = kChunks / kThreads;
#pragma unroll
  for (int i = 0; i <= kPer; ++i) {
    const int j = i * kThreads + (int)threadIdx.x;
    const int p0 = 8 * j - M;
    if (j > kChunks || p0 + 8 <= lo || p0 >= hi) continue;
    const u32x4 a = stage[stage_slot(j > 0 ? j - 1 : 0)];
    const u32x4 b = stage[stage_slot(j < kChunks ? j : kChunks - 1)];
    if (p0 >= lo && p0 + 8 <= hi) {
      __builtin_amdgcn_raw_buffer_store_b128(chunk_shifted<M>(a, b), a_r, j * 16, 0, kStreamStore);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int p = p0 + e;  // chunk j - 1 for e < M, chunk j from e = M
        if (p >= lo && p < hi) {
          const u32x4& c = e < M ? a : b;
          const int q = (e - M) & 7;
          o16[p] = (uint16_t)(c[q >> 1] >> (16 * (q & 1)));
        }
      }
    }
  }
}

// Block positions [lo, hi) of the chain's chunks to oblk, every thread of the
// workgroup (branches uniform).  A whole block on the 16-byte grid (kWhole: the
// launcher checked that) goes out in whole chunks, from registers where they
// leave the chain 1 KiB contiguous per wave (odd L); a partial block, or an
// output off that grid, is staged and stored in aligned 16-byte slots.
template <int L, int kBufs, bool kWhole = false, bool kDirect = L % 2 == 1>
__device__ __forceinline__ void store_block(const u32x4 (&v)[8], const Ctx& x, unsigned char* lds, __bf16* oblk,
                                            int lo, int hi) {
  if (kWhole || (lo == 0 && hi == kB && ((uintptr_t)oblk & 15) == 0)) {
    const auto out_r = rsrc(oblk, (uint32_t)(kB * 2));
    if constexpr (kDirect)
      store_direct(v, x, out_r);
    else
      store_staged(stage_chunks<L, kBufs, kDirect>(v, x, lds), out_r);
    return;
  }
  if constexpr (!kWhole) {
    const u32x4* stage = stage_chunks<L, kBufs, kDirect>(v, x, lds);
    if ((uintptr_t)oblk & 1) {  // not on the 2-byte grid: element stores
      uint16_t* o16 = reinterpret_cast<uint16_t*>(oblk);
      for (int p = lo + (int)threadIdx.x; p < hi; p += kThreads)
        o16[p] = reinterpret_cast<const uint16_t*>(stage + stage_slot(p >> 3))[p & 7];
      return;
    }
    switch (((uintptr_t)oblk >> 1) & 7) {
      case 0: store_range_shifted<0>(stage, oblk, lo, hi); break;
      case 1: store_range_shifted<1>(stage, oblk, lo, hi); break;
      case 2: store_range_shifted<2>(stage, oblk, lo, hi); break;
      case 3: store_range_shifted<3>(stage, oblk, lo, hi); break;
      case 4: store_range_shifted<4>(stage, oblk, lo, hi); break;
      case 5: store_range_shifted<5>(stage, oblk, lo, hi); break;
      case 6: store_range_shifted<6>(stage, oblk, lo, hi); break;
      default: store_range_shifted<7>(stage, oblk, lo, hi); break;
    }
  }
}

// A backward's partial row in whole 16-byte chunks up to its stride (a multiple
// of 8; the block sum reads only the first n values).
template <int L, int kBufs>
__device__ __forceinline__ void store_row(const u32x4 (&v)[8], const Ctx& x, unsigned char* lds, __bf16* row,
                                          uint32_t row_bytes) {
  const auto row_r = rsrc(row, row_bytes);
  if constexpr (L % 2 == 1)
    store_direct(v, x, row_r);
  else
    store_staged(stage_chunks<L, kBufs>(v, x, lds), row_r);
}

template <int L, bool kWhole, int kBufs>
__global__ __launch_bounds__(kThreads, kBufs == 1 ? 4 : 2) void bfht_mfma15_fwd(const __bf16* __restrict__ latent,
                                                            __bf16* __restrict__ out, int n,
                                                            int64_t first_block, int64_t start,
                                                            int64_t stop, uint32_t seed32) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(kBufs)];
  const int64_t block = first_block + blockIdx.x;
  const Ctx x = make_ctx(seed32, block);
  u32x4 src[kTiles][2];
  load_latent<kWhole>(x, latent, n, src);
  u32x4 v[8];
  // block-local output range [lo, hi); out element of block position p is (base - start) + p
  const int64_t base = block * kB;
  const int lo = kWhole ? 0 : (int)(start - base > 0 ? start - base : 0);
  const int hi = kWhole ? kB : (int)(stop - base < kB ? stop - base : kB);
  __bf16* oblk = out + (base - start);
  // A block that will be staged anyway does without layout F at odd L (a slice of 31
  // blocks off the 16-byte grid: 7.65 us against 7.92); two chains in one kernel need
  // more than the 128 registers of workgroups that share a CU.
  if constexpr (L % 2 == 1 && kBufs == 2 && !kWhole) {
    if (lo != 0 || hi != kB || ((uintptr_t)oblk & 15) != 0) {
      chain_chunks<L, kBufs, false>(x, lds, src, [](int i) { return i; }, v);
      store_block<L, kBufs, false, false>(v, x, lds, oblk, lo, hi);
      return;
    }
  }
  chain_chunks<L, kBufs>(x, lds, src, [](int i) { return i; }, v);
  store_block<L, kBufs, kWhole>(v, x, lds, oblk, lo, hi);
}

// ---------------------------------------------------------------- backward

// Loads block positions [lo, hi) of a block's gradient that starts M elements
// past a 16-byte boundary (gblk, 2-byte aligned), zero elsewhere: the chunk at
// positions p .. p + 7 is elements M .. 7 of aligned slot p / 8 followed by
// elements 0 .. M - 1 of the next slot.  A slot is read only when it holds
// positions of the range; the buffer spans the gradient's 16-byte granules
// (from the one holding its first element to the one holding its last, gend
// is one past it; at most the block's kChunks + 1 slots), so no read leaves
// them, and positions outside the range read from those granules are zeroed.
template <int M>
__device__ __forceinline__ void load_grad_shifted(const Ctx& x, const __bf16* gblk, const __bf16* gend, int lo,
                                                  int hi, u32x4 (&src)[kTiles][2]) {
  const uintptr_t a0 = (uintptr_t)gblk - 2 * M;
  const uintptr_t a1 = ((uintptr_t)gend + 15) & ~(uintptr_t)15;
  // every slot of the block lies in the first kChunks + 1 slots from a0
  const uintptr_t span = a1 - a0 < (uintptr_t)(kChunks + 1) * 16 ? a1 - a0 : (uintptr_t)(kChunks + 1) * 16;
  const auto g_r = rsrc((const void*)a0, (uint32_t)span);
  constexpr uint32_t kOff = 0x80000000u;
  load_source(
      x,
      [&](int p) -> u32x4 {
        const bool use_a = p + 7 - M >= lo && p < hi;            // slot p/8: positions p .. p + 7 - M
        const bool use_b = M > 0 && p + 7 >= lo && p + 8 - M < hi;  // next slot: p + 8 - M .. p + 7
        const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(g_r, (int)(use_a ? (uint32_t)(2 * p) : kOff), 0, 0);
        const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(g_r, (int)(use_b ? (uint32_t)(2 * p + 16) : kOff), 0, 0);
        u32x4 v = chunk_shifted<8 - M>(a, b);
        if (p < lo || p + 8 > hi) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (p + e < lo || p + e >= hi) v[e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
        }
        return v;
      },
      src);
}

// Source operands of one block's gradient: positions [lo, hi) of `gblk` (the
// block's position 0; `gend` is one past the whole gradient), zero elsewhere.
// kWhole: the whole block, 16-byte aligned.
__device__ __forceinline__ bool grad_whole(const __bf16* gblk, int lo, int hi) {
  return lo == 0 && hi == kB && ((uintptr_t)gblk & 15) == 0;
}
__device__ __forceinline__ void load_grad_whole(const Ctx& x, const __bf16* gblk, u32x4 (&src)[kTiles][2]) {
  const auto g_r = rsrc(gblk, (uint32_t)(kB * 2));
  load_source(x, [&](int p) -> u32x4 { return __builtin_amdgcn_raw_buffer_load_b128(g_r, p * 2, 0, 0); }, src);
}
template <bool kWhole>
__device__ __forceinline__ void load_grad(const Ctx& x, const __bf16* gblk, const __bf16* gend, int lo, int hi,
                                          u32x4 (&src)[kTiles][2]) {
  if (kWhole || grad_whole(gblk, lo, hi)) {  // uniform
    load_grad_whole(x, gblk, src);
    return;
  }
  if constexpr (!kWhole) {
    if ((uintptr_t)gblk & 1) {  // not on the 2-byte grid: element loads
      const uint16_t* gblk16 = reinterpret_cast<const uint16_t*>(gblk);
      load_source(
          x,
          [&](int p) -> u32x4 {
            u32x4 v = {0u, 0u, 0u, 0u};
            if (p + 8 > lo && p < hi) {
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (p + e >= lo && p + e < hi) v[e >> 1] |= (uint32_t)gblk16[p + e] << (16 * (e & 1));
            }
            return v;
          },
          src);
      return;
    }
    // part of a block, or a gradient off the 16-byte grid: aligned 16-byte slot loads
    switch (((uintptr_t)gblk >> 1) & 7) {
      case 0: load_grad_shifted<0>(x, gblk, gend, lo, hi, src); break;
      case 1: load_grad_shifted<1>(x, gblk, gend, lo, hi, src); break;
      case 2: load_grad_shifted<2>(x, gblk, gend, lo, hi, src); break;
      case 3: load_grad_shifted<3>(x, gblk, gend, lo, hi, src); break;
      case 4: load_grad_shifted<4>(x, gblk, gend, lo, hi, src); break;
      case 5: load_grad_shifted<5>(x, gblk, gend, lo, hi, src); break;
      case 6: load_grad_shifted<6>(x, gblk, gend, lo, hi, src); break;
      default: load_grad_shifted<7>(x, gblk, gend, lo, hi, src); break;
    }
  }
}

// Per-block partial latent gradient (first n positions) of the
// adjoint chain D_0 H D_1 ... H D_L applied to grad scattered into the block.
// The rows are bfloat16 (the gradient's own type; each of the ~2^8 terms of a
// position's sum carries one bf16 rounding, ~2^-9 relative, and the sum is
// formed in float32), half the traffic of float32 rows in both kernels.
// kWhole: every block's gradient is read whole from a 16-byte aligned place
// and n % 8 == 0 (the launcher checks), so no partial-chunk paths are needed.
template <int L, bool kWhole>
__global__ __launch_bounds__(kThreads, 2) void bfht_mfma15_bwd(const __bf16* __restrict__ grad,
                                                               __bf16* __restrict__ partial, int n,
                                                               int64_t first_block, int64_t start, int64_t stop,
                                                               uint32_t seed32) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(2)];
  const int64_t slot = blockIdx.x;
  const int64_t block = first_block + slot;
  const Ctx x = make_ctx(seed32, block);
  const int64_t base = block * kB;
  const int lo = kWhole ? 0 : (int)(start - base > 0 ? start - base : 0);
  const int hi = kWhole ? kB : (int)(stop - base < kB ? stop - base : kB);
  u32x4 src[kTiles][2];
  load_grad<kWhole>(x, grad + (base - start), grad + (stop - start), lo, hi, src);
  u32x4 v[8];
  chain_chunks<L, 2>(x, lds, src, [](int i) { return L - i; }, v);
  const int64_t stride = mfma15_part_stride(n);
  store_row<L, 2>(v, x, lds, partial + slot * stride, (uint32_t)stride * 2u);
}

// sum += the chain's result signed by its last sign layer, in the chain's end
// layout: F (odd L, words as direct_chunks reads them) or S0 (even L, words nw).
template <int L>
__device__ __forceinline__ void add_signed(f32x16 (&sum)[kTiles], const f32x16 (&acc)[kTiles], const Ctx& x,
                                           const uint32_t* words, const uint32_t (&nw)[4]) {
  // both dwords of `pair` shifted left: bit 31 of each is its own word's bit
  auto shl = [](uint64_t pair, int s) {
    uint64_t r;
    asm("v_lshlrev_b64 %0, %1, %2" : "=v"(r) : "s"(s), "v"(pair));
    return r;
  };
  auto add = [&](int t, int r, uint32_t m) {
    sum[t][r] += __uint_as_float(__float_as_uint(acc[t][r]) ^ (m & 0x80000000u));
  };
  if constexpr (L % 2 == 1) {
    const u32x4* wt = reinterpret_cast<const u32x4*>(words) + 2 * ((x.lane32 >> 1) + 16 * x.wave);
    const u32x4 wa = wt[0], wb = wt[1];
    const int sh = 4 * (x.l5 + 2 * (x.lane32 & 1));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint64_t pair = (uint64_t)(wa[k] >> sh) | ((uint64_t)(wb[k] >> sh) << 32);
#pragma unroll
      for (int j = 0; j < 8; ++j) {  // value j of chunks k and k + 4
        const uint64_t m = shl(pair, 31 - ((j >> 1) + 16 * (j & 1)));
        add(j & 3, (j >> 2) | (k << 1), (uint32_t)m);
        add(j & 3, 8 | (j >> 2) | (k << 1), (uint32_t)(m >> 32));
      }
    }
  } else {
    const uint64_t pair = (uint64_t)nw[0] | ((uint64_t)nw[1] << 32);  // p11 = 0, 1
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int r = 0; r < 8; ++r) {  // p0-1 = r bits 0-1, p4 = r bit 2, p2-3 = t
        const uint64_t m = shl(pair, 31 - ((r & 3) + 4 * t + 16 * (r >> 2)));
        add(t, r, (uint32_t)m);
        add(t, r + 8, (uint32_t)(m >> 32));
      }
  }
}

// The same over many blocks: workgroup g walks blocks g * group .. of the call in
// ascending order, adds their chains' results in float32 registers and stores
// one bfloat16 row, so a call of more blocks than CUs leaves about one row per
// CU for the block sum instead of one per block, and the next block's gradient
// loads while the current one transforms.  One workgroup per CU: the chain, the
// sum (64 registers) and the loads in flight (32) take up to 256 VGPRs.  The offsets
// of the loads of partial blocks, and of blocks off the 16-byte grid at each of its
// shifts, are the same for every block: the lane is hidden from the compiler before
// them, which would keep them all over the loop and spill 33 registers for it.  Three
// layers, block sum included, against a row per block (two workgroups per CU):
// 257 blocks 17.8 / 16.3 us, 300 18.1 / 18.4, 600 24.6 / 25.1, 1024 32.2 / 35.2,
// 2592 67 / 88 (of which the sum of 2592 rows takes 32); a gradient off the
// 16-byte grid, read without prefetch, 21.8 at 257 blocks, 29.0 at 513 and 91 at 2592
// (with the offsets kept 28.3, 37.2 and 127; a row per block and one workgroup per CU
// 24.3, 33.9 and 136).
template <int L, bool kWhole>
__device__ __forceinline__ void bwd_sum_row(const __bf16* __restrict__ grad, __bf16* __restrict__ row,
                                            int64_t stride, int64_t first_block, int64_t b0, int64_t b1,
                                            int64_t start, int64_t stop, uint32_t seed32, unsigned char* lds) {
  f32x16 sum[kTiles] = {};
  u32x4 next[kTiles][2];
  bool loaded = false;  // `next` holds the coming block (a whole, aligned one)
  Ctx x;
  for (int64_t b = b0; b < b1; ++b) {
    x = make_ctx(seed32, first_block + b);
    const int64_t base = (first_block + b) * kB;
    const __bf16* gblk = grad + (base - start);
    if (b > b0) __syncthreads();  // every wave has read the previous block's exchanges and words
    u32x4 src[kTiles][2];
    if (loaded) {
#pragma unroll
      for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) src[t][c] = next[t][c];
    } else {
      const int lo = kWhole ? 0 : (int)(start - base > 0 ? start - base : 0);
      const int hi = kWhole ? kB : (int)(stop - base < kB ? stop - base : kB);
      Ctx xl = x;
      if constexpr (!kWhole) asm volatile("" : "+v"(xl.lane32));  // see above
      load_grad<kWhole>(xl, gblk, grad + (stop - start), lo, hi, src);
    }
    // only the last block of a call can be partial after its first
    loaded = b + 1 < b1 && (kWhole || grad_whole(gblk + kB, 0, (int)(stop - base - kB < kB ? stop - base - kB : kB)));
    if (loaded) load_grad_whole(x, gblk + kB, next);
    f32x16 acc[kTiles];
    uint32_t nw[4];
    run_chain<L, L % 2 == 1, 2>(acc, x, lds, src, [](int i) { return L - i; }, nw);
    add_signed<L>(sum, acc, x, reinterpret_cast<const uint32_t*>(lds + 2 * kXBufBytes) + (L - 1) * kWordsPerLayer, nw);
  }
  u32x4 v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (L % 2 == 1) {  // direct_chunks' order
        const int r = (q >> 1) | (k << 1);
        v[k][q] = pk(sum[2 * (q & 1)][r], sum[2 * (q & 1) + 1][r]);
      } else {  // out_chunks' order
        const int t = (q >> 1) + 2 * (k & 1), r = 2 * (q & 1) + 4 * ((k >> 1) & 1) + 8 * (k >> 2);
        v[k][q] = pk(sum[t][r], sum[t][r + 1]);
      }
    }
  store_row<L, 2>(v, x, lds, row, (uint32_t)stride * 2u);
}

template <int L, bool kWhole>
__global__ __launch_bounds__(kThreads, 2) void bfht_mfma15_bwd_sum(const __bf16* __restrict__ grad,
                                                                   __bf16* __restrict__ partial, int n,
                                                                   int64_t first_block, int64_t nblocks,
                                                                   int64_t group, int64_t start, int64_t stop,
                                                                   uint32_t seed32) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(2)];
  const int64_t b0 = (int64_t)blockIdx.x * group, b1 = b0 + group < nblocks ? b0 + group : nblocks;
  const int64_t stride = mfma15_part_stride(n);
  bwd_sum_row<L, kWhole>(grad, partial + (int64_t)blockIdx.x * stride, stride, first_block, b0, b1, start, stop,
                         seed32, lds);
}

// ---------------------------------------------------------------- grouped


// Whole weight of each job (positions [0, size)): the chain of bfht_mfma15_fwd,
// the bf16 output times the job's weight scale.
template <int L, int kBufs>
__global__ __launch_bounds__(kThreads, kBufs == 1 ? 4 : 2) void bfht_mfma15_fwd_grouped(const GroupTable g) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(kBufs)];
  const int j = group_job(g, (int)blockIdx.x);
  const GroupJob& jb = g.job[j];
  const int64_t block = (int64_t)blockIdx.x - g.prefix[j];
  const Ctx x = make_ctx(jb.seed32, block);
  u32x4 src[kTiles][2];
  load_latent(x, static_cast<const __bf16*>(jb.src), jb.n, src);
  u32x4 v[8];
  chain_chunks<L, kBufs>(x, lds, src, [](int i) { return i; }, v, jb.scale);
  const int64_t base = block * kB;
  const int hi = jb.size - base < kB ? (int)(jb.size - base) : kB;
  store_block<L, kBufs>(v, x, lds, static_cast<__bf16*>(jb.dst) + base, 0, hi);
}

// Per-block partial rows of each job's whole-weight gradient (bf16 weight
// gradient, as bfht_mfma15_bwd), into the job's partial rows.
template <int L, int kBufs>
__global__ __launch_bounds__(kThreads, kBufs == 1 ? 4 : 2) void bfht_mfma15_bwd_grouped(const GroupTable g) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(kBufs)];
  const int j = group_job(g, (int)blockIdx.x);
  const GroupJob& jb = g.job[j];
  const int64_t slot = (int64_t)blockIdx.x - g.prefix[j];
  const Ctx x = make_ctx(jb.seed32, slot);
  const int64_t base = slot * kB;
  const int hi = jb.size - base < kB ? (int)(jb.size - base) : kB;
  const __bf16* g0 = static_cast<const __bf16*>(jb.src);
  u32x4 src[kTiles][2];
  load_grad<false>(x, g0 + base, g0 + jb.size, 0, hi, src);
  u32x4 v[8];
  chain_chunks<L, kBufs>(x, lds, src, [](int i) { return L - i; }, v);
  // the row stride is a multiple of 64
  store_row<L, kBufs>(v, x, lds, static_cast<__bf16*>(jb.part) + slot * (int64_t)jb.stride, (uint32_t)jb.stride * 2u);
}

// The same for jobs of more blocks than CUs, `run` blocks per row.
template <int L>
__global__ __launch_bounds__(kThreads, 2) void bfht_mfma15_bwd_sum_grouped(const GroupTable g) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[chain_lds_bytes(2)];
  const int j = group_job(g, (int)blockIdx.x);
  const GroupJob& jb = g.job[j];
  const int64_t index = (int64_t)blockIdx.x - g.prefix[j];
  const int64_t b0 = index * jb.run, b1 = b0 + jb.run < jb.nblocks ? b0 + jb.run : jb.nblocks;
  bwd_sum_row<L, false>(static_cast<const __bf16*>(jb.src),
                        static_cast<__bf16*>(jb.part) + index * (int64_t)jb.stride, jb.stride, 0, b0, b1, 0, jb.size,
                        jb.seed32, lds);
}

}  // namespace
}  // namespace mfma15

bool mfma15_applicable(const BfhtArgs& a, bool fwd) {
  // 16-byte vector loads of the latent and stores of the partial rows need
  // aligned bases; the backward reads the gradient in aligned 16-byte slots
  // whatever its offset, and output alignment is handled per block.
  const bool aligned = ((uintptr_t)a.src % (fwd ? 16 : 2) == 0) &&
                       (a.work == nullptr || (uintptr_t)a.work % 16 == 0);
  return a.dtype == kBF16 && a.log_block == mfma15::kLog && a.nblocks > 0 && a.n <= mfma15::kB && aligned;
}

namespace {

template <bool kWhole, int kBufs>
hipError_t launch_mfma15_fwd(const BfhtArgs& a, hipStream_t s) {
  using namespace mfma15;
  const dim3 grid((unsigned)a.nblocks), block(kThreads);
  auto* src = (const __bf16*)a.src;
  auto* dst = (__bf16*)a.dst;
  const int n = (int)a.n;
  switch (a.layers) {
    case 1: hipLaunchKernelGGL((bfht_mfma15_fwd<1, kWhole, kBufs>), grid, block, 0, s, src, dst, n, a.first_block, a.start, a.stop, a.seed32); break;
    case 2: hipLaunchKernelGGL((bfht_mfma15_fwd<2, kWhole, kBufs>), grid, block, 0, s, src, dst, n, a.first_block, a.start, a.stop, a.seed32); break;
    case 3: hipLaunchKernelGGL((bfht_mfma15_fwd<3, kWhole, kBufs>), grid, block, 0, s, src, dst, n, a.first_block, a.start, a.stop, a.seed32); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <bool kWhole>
hipError_t launch_mfma15_bwd(const BfhtArgs& a, hipStream_t s) {
  using namespace mfma15;
  const int64_t group = mfma15_bwd_group(a.nblocks);
  const dim3 grid((unsigned)mfma15_bwd_rows(a.nblocks)), block(kThreads);
  auto* src = (const __bf16*)a.src;
  auto* part = (__bf16*)a.work;  // bf16 partial rows (summed in float32, bfht_reduce_blocks)
  const int n = (int)a.n;
#define LWL_BWD(L)                                                                                               \
  if (group > 1)                                                                                                 \
    hipLaunchKernelGGL((bfht_mfma15_bwd_sum<L, kWhole>), grid, block, 0, s, src, part, n, a.first_block,        \
                       a.nblocks, group, a.start, a.stop, a.seed32);                                             \
  else                                                                                                           \
    hipLaunchKernelGGL((bfht_mfma15_bwd<L, kWhole>), grid, block, 0, s, src, part, n, a.first_block, a.start,   \
                       a.stop, a.seed32)
  switch (a.layers) {
    case 1: LWL_BWD(1); break;
    case 2: LWL_BWD(2); break;
    case 3: LWL_BWD(3); break;
    default: return hipErrorInvalidValue;
  }
#undef LWL_BWD
  return hipGetLastError();
}

}  // namespace

hipError_t launch_mfma15_grouped(const GroupTable& g, int layers, hipStream_t s, bool fwd, bool summed) {
  using namespace mfma15;
  if (g.count <= 0 || g.prefix[g.count] == 0) return hipSuccess;
  const dim3 grid((unsigned)g.prefix[g.count]), block(kThreads);
  const bool paired = chains_share_cu(g.prefix[g.count]);
#define LWL_GROUPED(L)                                                                      \
  if (fwd && paired)                                                                        \
    hipLaunchKernelGGL((bfht_mfma15_fwd_grouped<L, 1>), grid, block, 0, s, g);              \
  else if (fwd)                                                                             \
    hipLaunchKernelGGL((bfht_mfma15_fwd_grouped<L, 2>), grid, block, 0, s, g);              \
  else if (summed)                                                                          \
    hipLaunchKernelGGL((bfht_mfma15_bwd_sum_grouped<L>), grid, block, 0, s, g);             \
  else if (paired)                                                                          \
    hipLaunchKernelGGL((bfht_mfma15_bwd_grouped<L, 1>), grid, block, 0, s, g);              \
  else                                                                                      \
    hipLaunchKernelGGL((bfht_mfma15_bwd_grouped<L, 2>), grid, block, 0, s, g)
  switch (layers) {
    case 1: LWL_GROUPED(1); break;
    case 2: LWL_GROUPED(2); break;
    case 3: LWL_GROUPED(3); break;
    default: return hipErrorInvalidValue;
  }
#undef LWL_GROUPED
  return hipGetLastError();
}

hipError_t launch_mfma15(const BfhtArgs& a, hipStream_t s, bool fwd) {
  using namespace mfma15;
  // whole blocks: [start, stop) covers exactly blocks first_block .. +nblocks, and the
  // slice base (out / grad) is 16-byte aligned, so every block's base is too
  const bool whole = a.start == a.first_block * kB && a.stop == (a.first_block + a.nblocks) * kB &&
                     (uintptr_t)a.dst % 16 == 0 && (uintptr_t)a.src % 16 == 0 && a.n % 8 == 0;
  if (!fwd) return whole ? launch_mfma15_bwd<true>(a, s) : launch_mfma15_bwd<false>(a, s);
  if (chains_share_cu(a.nblocks)) return whole ? launch_mfma15_fwd<true, 1>(a, s) : launch_mfma15_fwd<false, 1>(a, s);
  return whole ? launch_mfma15_fwd<true, 2>(a, s) : launch_mfma15_fwd<false, 2>(a, s);
}

}  // namespace lwl
