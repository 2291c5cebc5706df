// Fused BlockFHTLinear forward for the reference extension's own domain:
// float32 / float16 / bfloat16, block B <= 2^14 and B % in_features == 0
// (reference gate latent_weight_lab/block_fht.py:263-273, kernel
// csrc/block_fht_ext_cuda.cu:225-329, launcher :624-681).
//
// out[t, o] = sum_i x[t, i] * (weight_scale * W[o, i]),  W[o, i] = y[o * in + i]
//
// in_features divides B, so every output row lies inside one generated block
// and no row straddles two.  A workgroup owns G consecutive blocks (the slots of
// the whole-block VALU generator: one block of 2^14 per 512-thread workgroup,
// or 256 / (B/32) smaller blocks per 256-thread workgroup) and a range of
// tokens.  It generates its blocks in float32 straight into an LDS weight tile
// (the generator's final stores land in LDS instead of memory, over its own
// exchange buffers once every thread has read them, already scaled
// by weight_scale, as the reference scales its shared-memory values), then
// contracts the tile with its tokens: a team of min(in, 64) lanes computes four
// tokens of one output row, lanes striding over k, and sums its lanes with
// butterfly shuffles.  All arithmetic is float32; x and out keep the I/O type.
// The weight never touches memory.
#include "bfht_block.h"

#include <vector>

namespace lwl {
namespace {

// LDS window of the generator's stores: global position g of the workgroup's
// tile lands at w[g - base], multiplied by weight_scale.  `range` / call take
// the role of the buffer-resource form of the per-block store (indices outside
// [0, count) are dropped), `at` the element form.
struct LdsRange {
  int first;
  int count;
};
struct LdsWeightStore {
  float* w;
  int64_t base;
  float scale;
  __device__ LdsRange range(int64_t first, int64_t count) const {
    return LdsRange{(int)(first - base), (int)count};
  }
  __device__ void operator()(LdsRange r, int i, float v) const {
    if ((unsigned)i < (unsigned)r.count) w[r.first + i] = v * scale;
  }
  __device__ void whole(LdsRange r, int b, int c, float v) const { w[r.first + b + c] = v * scale; }
  __device__ void at(int64_t i, float v) const { w[i - base] = v * scale; }
};

constexpr int kQuad = 4;  // tokens per team pass
constexpr int kSpan = 8;  // k iterations of a lane whose x loads are in flight together

// LDS of a workgroup.  Narrow: the generator's exchange buffers and sign tables,
// then (over them, once they are read) the weight tile and the staged x of one
// token quad, 4096 values of it, so that a 2^14 block takes 80 KiB and two
// workgroups share a CU.  Wide: the weight tile behind the generator's LDS, which
// holds a single token's staged x afterwards; one workgroup per CU at 2^14, two
// below, and no barrier before the tile's stores.
constexpr int kQuadStage = 4096;
template <int LB, bool kWide>
struct SmallLinearGeo {
  using Gm = Geo<LB>;
  static constexpr int kTileElems = Gm::G * Gm::B;  // weights generated per workgroup
  static constexpr int kStage = kWide ? BlockLds<LB>::FLOATS : kQuadStage;
  static_assert(!kWide || kStage >= Gm::B, "one token's row fits the generator's LDS");
  static constexpr int kTile = kWide ? BlockLds<LB>::FLOATS : 0;   // where the weight tile starts
  static constexpr int kStaged = kWide ? 0 : kTileElems;           // and the staged x
  static constexpr int kNeed = kTileElems + kStage;
  static constexpr int kLdsFloats = kNeed > BlockLds<LB>::FLOATS ? kNeed : BlockLds<LB>::FLOATS;
  static_assert(kLdsFloats * 4 <= 160 * 1024 && (kWide || LB > 14 || kLdsFloats * 8 <= 160 * 1024), "LDS of one CU");
};
// staged values of a token quad: one token's when the call has only one
__host__ __device__ constexpr int64_t small_stage(int64_t tokens, int64_t in_f) { return (tokens == 1 ? 1 : kQuad) * in_f; }

template <int LB, class T, bool kWide>
__device__ __forceinline__ void small_item(const T* __restrict__ x, const T* __restrict__ latent, T* __restrict__ out,
                                           int tokens, int in_f, int log_in, int out_f, int n, int64_t nblocks,
                                           uint32_t seed32, int layers, float scale, int token_split, int64_t tile,
                                           int split, const LinearEpi& ep, float* smem) {
  using Gm = Geo<LB>;
  using SG = SmallLinearGeo<LB, kWide>;
  float* wt = smem + SG::kTile;  // the weight tile, row-major [rows][in]
  const int64_t size = (int64_t)in_f * out_f;
  const int64_t base = tile * SG::kTileElems;

  // this split's token quads, and the x of a quad staged in LDS (step 2)
  const int quads = (tokens + kQuad - 1) / kQuad;
  const int per_split = (quads + token_split - 1) / token_split;
  const int q0 = split * per_split;
  const int q1 = q0 + per_split < quads ? q0 + per_split : quads;
  const auto x_r = tile_rsrc(x, (uint64_t)tokens * in_f * sizeof(T));
  const int nstage = (int)small_stage(tokens, in_f);
  const bool staged = kWide ? tokens == 1 : nstage <= SG::kStage;
  // thread's share i0 + e * WG (e < kSpan) of quad q's staged x (tokens past the batch read 0)
  auto stage_load = [&](int q, int i0, float (&v)[kSpan]) {
#pragma unroll
    for (int e = 0; e < kSpan; ++e) {
      const int i = i0 + e * Gm::WG;
      const int t = q * kQuad + (i >> log_in);
      v[e] = buf_load<T>(x_r, i < nstage && t < tokens ? t * in_f + (i & (in_f - 1)) : -1);
    }
  };
  // When one round of loads stages a quad, the first quad's are issued before
  // the generator runs, which hides their latency.
  const bool prefetch = staged && nstage <= kSpan * Gm::WG && q0 < q1;
  float xpre[kSpan];
  if (prefetch) stage_load(q0, (int)threadIdx.x, xpre);

  // 1. the tile's G blocks (inactive slots past the last block store nothing;
  //    their rows lie past out_features and are never read)
  const int64_t slot = tile * Gm::G + (threadIdx.x >> Gm::LT);
  block_fwd_slot<LB, T, Gm::G, !kWide>(latent, LdsWeightStore{wt, base, scale}, n, 0, slot, nblocks, 0, size, seed32,
                                     layers, smem);
  __syncthreads();

  // 2. rows row0 .. row0 + rows - 1 against this split's token quads
  const int row0 = (int)(base >> log_in);
  const int tile_rows = SG::kTileElems >> log_in;
  const int rows = out_f - row0 < tile_rows ? out_f - row0 : tile_rows;
  if (rows <= 0 || q0 >= q1) return;  // uniform across the workgroup
  const int log_ks = log_in < 6 ? log_in : 6;  // lanes per team: min(in, 64)
  const int ks = 1 << log_ks;
  const int lane = threadIdx.x & 63;
  const int j = lane & (ks - 1);
  const int team = (int)(threadIdx.x >> log_ks);
  const int nteams = Gm::WG >> log_ks;
  const int npairs = (q1 - q0) * rows;
  const auto o_r = tile_rsrc(out, (uint64_t)tokens * out_f * sizeof(T));
  // epilogue terms (uniform); absent inputs get empty resources
  const bool has_xs = ep.xsum != nullptr, has_base = ep.base != nullptr, has_bias = ep.bias != nullptr;
  const float cx = has_xs ? ep.cscale * *ep.coef : 0.f;
  const auto xs_r = tile_rsrc(has_xs ? (const void*)ep.xsum : (const void*)out, has_xs ? (uint64_t)tokens * 4 : 0);
  const auto b_r = tile_rsrc(has_base ? ep.base : (const void*)out, has_base ? (uint64_t)tokens * out_f * sizeof(T) : 0);
  const auto bias_r = tile_rsrc(has_bias ? ep.bias : (const void*)out, has_bias ? (uint64_t)out_f * sizeof(T) : 0);
  // One team pass: rows r, r + rstride, ... (NR of them; those from `rows` on
  // compute on row r and store nothing) against the first NU tokens of quad q
  // (NU = 1 for a quad holding one token, else kQuad).  Lane j adds
  // x[t][k] w[row][k] for k = j, j + ks, ... in that order (x from `xat`),
  // then the team's lanes are summed with butterfly shuffles.  A team's lanes
  // share the pass, so the shuffles only read lanes that run the same
  // iteration.  Every (row, token) sum takes the same additions in the same
  // order whatever NR and NU are.
  auto pass = [&](auto nr_c, auto nu_c, int q, int r, int rstride, auto xat) {
    constexpr int NR = decltype(nr_c)::value, NU = decltype(nu_c)::value;
    const int t0 = q * kQuad;
    const float* wrow[NR];
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int rh = r + h * rstride;
      wrow[h] = wt + ((rh < rows ? rh : r) << log_in);
    }
    float acc[NR][NU];
#pragma unroll
    for (int h = 0; h < NR; ++h)
#pragma unroll
      for (int u = 0; u < NU; ++u) acc[h][u] = 0.f;
    // kSpan iterations' loads are issued before their products (the loop's
    // trip count is not known at compile time, so without this each iteration
    // waited out one load's latency); the k order is the same either way
    int k = j;
    for (; k + (kSpan - 1) * ks < in_f; k += kSpan * ks) {
      float xv[kSpan][NU], wv[kSpan][NR];
#pragma unroll
      for (int i = 0; i < kSpan; ++i) {
#pragma unroll
        for (int h = 0; h < NR; ++h) wv[i][h] = wrow[h][k + i * ks];
#pragma unroll
        for (int u = 0; u < NU; ++u) xv[i][u] = xat(t0, u, k + i * ks);
      }
#pragma unroll
      for (int i = 0; i < kSpan; ++i)
#pragma unroll
        for (int h = 0; h < NR; ++h)
#pragma unroll
          for (int u = 0; u < NU; ++u) acc[h][u] += xv[i][u] * wv[i][h];
    }
    for (; k < in_f; k += ks) {
#pragma unroll
      for (int h = 0; h < NR; ++h) {
        const float w = wrow[h][k];
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[h][u] += xat(t0, u, k) * w;
      }
    }
    // the lane sums: each distance's shuffles of every sum in flight together
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) {
      if (s >= ks) continue;  // uniform
      float sh[NR][NU];
#pragma unroll
      for (int h = 0; h < NR; ++h)
#pragma unroll
        for (int u = 0; u < NU; ++u) sh[h][u] = __shfl_xor(acc[h][u], s, 64);
#pragma unroll
      for (int h = 0; h < NR; ++h)
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[h][u] += sh[h][u];
    }
    if (j == 0) {
      // The epilogue's inputs first, none behind a branch on its term or
      // behind a store that may alias it (either would be waited out on its
      // own): an absent term's buffer is empty and reads 0, and so does index
      // -1 (rows from `rows` on, tokens past the batch), whose store is dropped.
      float xs[NU], bias_o[NR], base_v[NR][NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) xs[u] = cx * buf_load<float>(xs_r, t0 + u < tokens ? t0 + u : -1);
#pragma unroll
      for (int h = 0; h < NR; ++h) {
        const int rh = r + h * rstride, o = row0 + rh;
        bias_o[h] = buf_load<T>(bias_r, rh < rows ? o : -1);
#pragma unroll
        for (int u = 0; u < NU; ++u)
          base_v[h][u] = buf_load<T>(b_r, rh < rows && t0 + u < tokens ? (t0 + u) * out_f + o : -1);
      }
#pragma unroll
      for (int h = 0; h < NR; ++h) {
        const int rh = r + h * rstride;
        if (rh >= rows) continue;  // uniform across the team
        const int o = row0 + rh;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int t = t0 + u;
          const int i = t < tokens ? t * out_f + o : -1;  // -1: the store is dropped
          buf_store<T>(linear_epilogue(acc[h][u], has_xs, xs[u], has_base, base_v[h][u], has_bias, bias_o[h]), o_r, i);
        }
      }
    }
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  using Quad = std::integral_constant<int, kQuad>;
  if (staged) {
    // Each quad's x rows are staged once and every team reads them there: read
    // from memory, all the workgroup's passes (and all the workgroups of an XCD,
    // at decode batches) ask its L2 for the same few lines.  Tokens past the
    // batch stage as 0.
    float* xs = smem + SG::kStaged;
    for (int q = q0; q < q1; ++q) {
      if (q > q0) __syncthreads();  // every team has read the previous quad
      for (int i0 = (int)threadIdx.x; i0 < nstage; i0 += kSpan * Gm::WG) {
        float v[kSpan];
        if (prefetch && q == q0) {
#pragma unroll
          for (int e = 0; e < kSpan; ++e) v[e] = xpre[e];
        } else {
          stage_load(q, i0, v);
        }
#pragma unroll
        for (int e = 0; e < kSpan; ++e)
          if (i0 + e * Gm::WG < nstage) xs[i0 + e * Gm::WG] = v[e];
      }
      __syncthreads();
      // two rows per pass (x read once for both); a quad of one token (decode)
      // computes that token alone
      auto xat = [&](int, int u, int kk) { return xs[(u << log_in) + kk]; };
      const bool single = tokens - q * kQuad == 1;
      for (int r = team; r < rows; r += 2 * nteams) {
        if (single)
          pass(Two{}, One{}, q, r, nteams, xat);
        else
          pass(Two{}, Quad{}, q, r, nteams, xat);
      }
    }
  } else {
    for (int pr = team; pr < npairs; pr += nteams) {
      const int q = q0 + pr / rows;
      int xi[kQuad];
#pragma unroll
      for (int u = 0; u < kQuad; ++u) xi[u] = q * kQuad + u < tokens ? (q * kQuad + u) * in_f : -1;  // -1: reads 0
      pass(One{}, Quad{}, q, pr - (pr / rows) * rows, 0,
           [&](int, int u, int kk) { return buf_load<T>(x_r, xi[u] < 0 ? -1 : xi[u] + kk); });
    }
  }
}

template <int LB, class T, bool kWide>
__global__ __launch_bounds__(Geo<LB>::WG) void bfht_linear_small(const T* __restrict__ x,
                                                                 const T* __restrict__ latent, T* __restrict__ out,
                                                                 int tokens, int in_f, int log_in, int out_f, int n,
                                                                 int64_t nblocks, uint32_t seed32, int layers,
                                                                 float scale, int token_split, LinearEpi ep) {
  __shared__ float smem[SmallLinearGeo<LB, kWide>::kLdsFloats];
  small_item<LB, T, kWide>(x, latent, out, tokens, in_f, log_in, out_f, n, nblocks, seed32, layers, scale, token_split,
                           blockIdx.x, (int)blockIdx.y, ep, smem);
}

// Several matrices in one launch (decode): workgroup i serves job j with
// prefix[j] <= i < prefix[j + 1], tile i - prefix[j] of it, all of its tokens.
// One matrix is one workgroup per CU, most of whose time is the generator's
// exchanges and barriers; together two workgroups share each CU and no launch
// waits for the last one's slowest workgroup (16 float32 matrices 1024 -> 4096,
// blocks of 2^14, two layers: 181 -> 113 us at one token, 205 -> 122 at 4, 351 ->
// 204 at 12; 24 matrices of 64 x 256 weights, one workgroup each: 451 -> 27).
template <int LB, class T>
__global__ __launch_bounds__(Geo<LB>::WG, 4) void bfht_linear_small_grouped(const SmallGroupTable g) {
  __shared__ float smem[SmallLinearGeo<LB, false>::kLdsFloats];
  const int j = group_job(g, (int)blockIdx.x);
  const SmallGroupJob& jb = g.job[j];
  const LinearEpi ep{jb.bias, jb.base, nullptr, nullptr, 0.f};
  small_item<LB, T, false>((const T*)jb.x, (const T*)jb.latent, (T*)jb.out, jb.tokens, 1 << jb.log_in, jb.log_in,
                           jb.out_f, jb.n, jb.nblocks, jb.seed32, jb.layers, jb.scale, 1,
                           (int64_t)blockIdx.x - g.prefix[j], 0, ep, smem);
}

// Float32 sums of the rows of x (the fused linear's row-sum term): one wave per
// row, lanes striding over k with eight loads in flight, then a fixed butterfly.
template <class T>
__global__ __launch_bounds__(256) void bfht_row_sums(const T* __restrict__ x, int tokens, int in_f,
                                                     float* __restrict__ xsum) {
  const int t = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // scalar: uniform resource
  if (t >= tokens) return;
  const int lane = threadIdx.x & 63;
  const auto x_r = tile_rsrc(x + (int64_t)t * in_f, (uint64_t)in_f * sizeof(T));  // k >= in_f reads 0
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < in_f; k0 += 8 * 64) {
#pragma unroll
    for (int u = 0; u < 8; ++u) s[u] += buf_load<T>(x_r, k0 + 64 * u + lane);
  }
  float v = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  if (lane == 0) xsum[t] = v;
}

int log2_of(int64_t v) {
  int l = 0;
  while (((int64_t)1 << l) < v) ++l;
  return l;
}

template <int LB, class T>
hipError_t launch_small_lb(const LinearArgs& a, hipStream_t s) {
  using Gm = Geo<LB>;
  const int64_t wtiles = (a.nblocks_w + Gm::G - 1) / Gm::G;
  const int log_in = log2_of(a.in_features);
  // The narrow form wherever it stages a quad's x, but for a single token under at most one
  // workgroup per CU, which gain nothing from a second and take the wide form, without the
  // narrow one's barrier before the stores (float16 1024 -> 4096: 12.2 -> 11.7 us; with more
  // tokens the narrow form is as fast or faster).  A longer row is staged alone (one
  // token, wide: 16384 -> 1000 in float32 107 -> 65 us) or read by every team from the
  // caches (several tokens): with a quad staged in rounds its loads were waited out
  // between barriers (4096 -> 1000, 1000 tokens: float32 1981 -> 715 us, float16 2034 ->
  // 772).  Of those calls the wide form takes the ones that fit one workgroup per CU,
  // which gain nothing from the second (16384 -> 64, 16 tokens: 30.4 against 33.9 us; 8192
  // -> 1000, 15 tokens, 500 workgroups: 47 against 37), and float32 calls whose x no longer
  // stays in the last-level cache while many rounds of workgroups stream it: twice as
  // many drift twice as far apart (16384 -> 4096: 512 tokens, 32 MiB, 7.3 against 5.6 ms;
  // 1000 tokens 14.1 against 24.7; 4003 tokens 57 against 125.  4096 -> 10000: 4003 tokens
  // 36 against 29; 8000 tokens 72 against 85.  The line keeps every measured call from losing, at the
  // price of a few that would still gain).  float16 keeps its lead to 2^29 bytes of x.
  const int64_t nstage = small_stage(a.tokens, a.in_features);
  const bool one_per_cu = wtiles * a.token_splits <= device_cus();
  const bool streams_x = sizeof(T) == 4 && a.tokens * a.in_features * 4 >= ((int64_t)48 << 20) &&
                         (double)(a.tokens * a.in_features) * (double)(a.in_features * a.out_features) >= 5e14;
  const bool wide = LB > 10 && (nstage > kQuadStage ? a.tokens == 1 || one_per_cu || streams_x
                                                    : a.tokens == 1 && one_per_cu);
#define LWL_SMALL(W)                                                                                                \
  hipLaunchKernelGGL((bfht_linear_small<LB, T, W>), dim3((unsigned)wtiles, (unsigned)a.token_splits), dim3(Gm::WG), \
                     0, s, (const T*)a.x, (const T*)a.latent, (T*)a.out, (int)a.tokens, (int)a.in_features, log_in, \
                     (int)a.out_features, (int)a.n, a.nblocks_w, a.seed32, a.layers, a.weight_scale,                \
                     a.token_splits, a.epi)
  if (wide)
    LWL_SMALL((LB > 10));
  else
    LWL_SMALL(false);
#undef LWL_SMALL
  return hipGetLastError();
}

template <int LB, class T>
hipError_t launch_small_grouped_lb(const LinearArgs* const* jobs, int count, hipStream_t s) {
  using Gm = Geo<LB>;
  SmallGroupTable g{};
  g.count = count;
  int64_t wg = 0;
  for (int i = 0; i < count; ++i) {
    const LinearArgs& a = *jobs[i];
    SmallGroupJob& jb = g.job[i];
    jb.x = a.x;
    jb.latent = a.latent;
    jb.out = a.out;
    jb.bias = a.epi.bias;
    jb.base = a.epi.base;
    jb.tokens = (int)a.tokens;
    jb.log_in = log2_of(a.in_features);
    jb.out_f = (int)a.out_features;
    jb.n = (int)a.n;
    jb.nblocks = (int)a.nblocks_w;
    jb.layers = a.layers;
    jb.seed32 = a.seed32;
    jb.scale = a.weight_scale;
    g.prefix[i] = (int)wg;
    wg += (a.nblocks_w + Gm::G - 1) / Gm::G;
  }
  g.prefix[count] = (int)wg;
  hipLaunchKernelGGL((bfht_linear_small_grouped<LB, T>), dim3((unsigned)wg), dim3(Gm::WG), 0, s, g);
  return hipGetLastError();
}

template <class T, int... LBs>
hipError_t dispatch_small(const LinearArgs& a, hipStream_t s, std::integer_sequence<int, LBs...>) {
  using Fn = hipError_t (*)(const LinearArgs&, hipStream_t);
  static const Fn table[] = {&launch_small_lb<LBs, T>...};
  return table[a.log_block](a, s);
}

template <class T, int... LBs>
hipError_t dispatch_small_grouped(int log_block, const LinearArgs* const* jobs, int count, hipStream_t s,
                                  std::integer_sequence<int, LBs...>) {
  using Fn = hipError_t (*)(const LinearArgs* const*, int, hipStream_t);
  static const Fn table[] = {&launch_small_grouped_lb<LBs, T>...};
  return table[log_block](jobs, count, s);
}

}  // namespace

bool linear_small_applicable(int dtype, int log_block, int64_t in_features) {
  if (dtype != kF32 && dtype != kF16 && dtype != kBF16) return false;
  if (log_block < 0 || log_block > kLinearSmallMaxLog || in_features <= 0) return false;
  return (((int64_t)1 << log_block) % in_features) == 0;
}

int linear_small_token_splits(const LinearArgs& a) {
  // Each split regenerates the workgroup's blocks: at least 32 token quads
  // (128 tokens) per split, and no more workgroups than about four per CU.
  const int g = a.log_block >= 5 ? (a.log_block >= 13 ? 1 : 256 >> (a.log_block - 5)) : 256;
  const int64_t wtiles = (a.nblocks_w + g - 1) / g;
  const int64_t quads = (a.tokens + kQuad - 1) / kQuad;
  int64_t split = (quads + 31) / 32;
  const int64_t cap = wtiles >= 1024 ? 1 : (1024 + wtiles - 1) / wtiles;
  if (split > cap) split = cap;
  if (split > 65535) split = 65535;
  return (int)(split < 1 ? 1 : split);
}

bool linear_small_groupable(const LinearArgs& a) {
  // calls of one token range whose staged quad fits the narrow form; their block
  // count and tile count stay far below 2^31 (tokens * out and in * out do)
  return linear_small_applicable(a.dtype, a.log_block, a.in_features) && !linear_small_mm_applicable(a) &&
         a.token_splits == 1 && a.nblocks_w < ((int64_t)1 << 24) &&
         small_stage(a.tokens, a.in_features) <= kQuadStage;
}

hipError_t launch_linear_small_grouped(const LinearArgs* jobs, int64_t count, hipStream_t s) {
  // one launch per (type, block size) of up to kSmallGroupMax jobs, buckets in
  // order of their first job
  using Seq = std::make_integer_sequence<int, kLinearSmallMaxLog + 1>;
  std::vector<bool> done((size_t)count, false);
  std::vector<const LinearArgs*> bucket;
  for (int64_t i = 0; i < count; ++i) {
    if (done[(size_t)i]) continue;
    bucket.clear();
    for (int64_t k = i; k < count && (int)bucket.size() < kSmallGroupMax; ++k)
      if (!done[(size_t)k] && jobs[k].dtype == jobs[i].dtype && jobs[k].log_block == jobs[i].log_block) {
        done[(size_t)k] = true;
        bucket.push_back(&jobs[k]);
      }
    hipError_t e = hipErrorInvalidValue;
    const int lb = jobs[i].log_block, m = (int)bucket.size();
    switch (jobs[i].dtype) {
      case kF32: e = dispatch_small_grouped<float>(lb, bucket.data(), m, s, Seq{}); break;
      case kF16: e = dispatch_small_grouped<f16>(lb, bucket.data(), m, s, Seq{}); break;
      case kBF16: e = dispatch_small_grouped<bf16>(lb, bucket.data(), m, s, Seq{}); break;
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_row_sums(const LinearArgs& a, float* xsum, hipStream_t s) {
  if (a.tokens == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.tokens + 3) / 4)), block(256);
  switch (a.dtype) {
    case kF32: hipLaunchKernelGGL(bfht_row_sums<float>, grid, block, 0, s, (const float*)a.x, (int)a.tokens,
                                  (int)a.in_features, xsum); break;
    case kF16: hipLaunchKernelGGL(bfht_row_sums<f16>, grid, block, 0, s, (const f16*)a.x, (int)a.tokens,
                                  (int)a.in_features, xsum); break;
    case kBF16: hipLaunchKernelGGL(bfht_row_sums<bf16>, grid, block, 0, s, (const bf16*)a.x, (int)a.tokens,
                                   (int)a.in_features, xsum); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_linear_small(const LinearArgs& a, hipStream_t s) {
  using Seq = std::make_integer_sequence<int, kLinearSmallMaxLog + 1>;
  switch (a.dtype) {
    case kF32: return dispatch_small<float>(a, s, Seq{});
    case kF16: return dispatch_small<f16>(a, s, Seq{});
    case kBF16: return dispatch_small<bf16>(a, s, Seq{});
  }
  return hipErrorInvalidValue;
}

}  // namespace lwl
