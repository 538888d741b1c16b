// Prefill path: the routed experts of a whole chunk, grouped by expert (each expert's weights
// are decoded once per tile of its tokens), on the fp8 MFMA.
//
//   grouped_hist     per chunk of routes: the count of each expert, and `run` (token t's routes are
//                    entries t k .. t k + k - 1 of `ord`) and a no-slot mark in `ord` for a route
//                    naming no expert of the layer
//   grouped_plan     one workgroup: per-expert counts (summed over the chunks, or from a slot list the
//                    caller built), exclusive scan, tile lists
//   grouped_place    per chunk: its (token, route) pairs in token order (stable), so every slot and
//                    every output sum has a fixed order; writes the slot list (token, weight and
//                    activation exponent per slot, `ord`: each token's slots in route order)
//   grouped_plan_small  these three in one workgroup, for at most kSmallPairs routes
//   grouped_prep_x   per token: exponent and E4M3 terms of the activation (2 terms for a bf16
//                    input: exact for every element of at least 2^-13 of the token's largest
//                    magnitude, where both terms are normal E4M3 numbers, and within 2^-20 of that
//                    maximum below it; 3 when a low bf16 term is given)
//   (each GEMM runs once per width class of its tiles, kClsCT, in an instantiation whose MFMAs,
//   fragment reads and direct loads cover just the class's columns)
//   grouped_gemm<0>  gate/up: (row block of 128 inter rows, token tile): 8 waves x 16 rows of
//                    gate and the same 16 of up, K = hidden in 128-column MFMA steps, 12 column
//                    tiles per A fragment; epilogue combines terms, applies row scales, SwiGLU,
//                    writes the activation as terms
//   grouped_gemm<1>  down: (row block of 256 hidden rows, slot tile): 8 waves x 32 rows, same
//                    structure over K = inter, writes each slot's unweighted down output z[slot]
//   grouped_combine  y[t] (+)= sum over token t's slots in `ord` order of wt[slot] * z[slot]
//
// Reference counterparts: run_batch_device's prefill arm (src/gpu/static_placement.hip:
// 1348-1964): moe_plan_kernel (src/gpu/moe_plan.hip:116-380), batch_quant_fp8_kernel
// (src/gpu/batch_kernels.hip:146-211), expert_gemm_wmma_kernel (src/gpu/expert_kernel.hip:
// 364-825), expert_swiglu_quant_kernel (862-931), expert_scatter_slots_kernel (935-947).
#include "affx_lut.h"

namespace affx {

constexpr int kPlanThreads = 1024;

struct Tile {
  uint32_t expert, slot0, n;
};

// Tiles of each GEMM by width class, kClsCT[k] column tiles of tokens: an expert's full tiles and a
// partial last one in the narrowest class that holds its tokens, stored widest class first; each
// class runs in its own instantiation of the GEMM.
constexpr int kNCls = 4;
constexpr int kClsCT[kNCls] = {12, 8, 4, 2};
__host__ __device__ inline uint32_t cls_ct(uint32_t k) {
  uint32_t ct = kClsCT[0];
  for (uint32_t q = 1; q < (uint32_t)kNCls; ++q)
    if (q == k) ct = kClsCT[q];
  return ct;
}
struct GroupedHdr {
  uint32_t n_slots;
  uint32_t tx;                     // activation terms of the gate/up input (2 or 3)
  uint32_t bad;                    // a caller's slot list needed more tiles than it can hold
  uint32_t n_cls[2][kNCls];        // [GEMM][class] tile counts
};

// ------------------------------------------------------------------------------------------------
// plan
// ------------------------------------------------------------------------------------------------
// Exclusive scan over the workgroup (kPlanThreads threads, thread i holds v[i]) of N counts at
// once; returns thread i's prefixes and writes the totals to tot.
template <int N>
__device__ __forceinline__ void plan_scan(uint32_t (&v)[N], uint32_t* wsum, uint32_t (&tot)[N]) {
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  constexpr uint32_t kW = kPlanThreads / 64;
  uint32_t inc[N];
#pragma unroll
  for (int q = 0; q < N; ++q) inc[q] = v[q];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1)
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const uint32_t n = __shfl_up(inc[q], o);
      if (lane >= (uint32_t)o) inc[q] += n;
    }
  if (lane == 63)
#pragma unroll
    for (int q = 0; q < N; ++q) wsum[q * kW + wv] = inc[q];
  __syncthreads();
  // the waves' totals: scanned by one 16-lane run per count
  static_assert(kW == 16 && N * kW <= kPlanThreads, "");
  const uint32_t x = tid < N * kW ? wsum[tid] : 0u;
  uint32_t in = x;
#pragma unroll
  for (int o = 1; o < (int)kW; o <<= 1) {
    const uint32_t n = __shfl_up(in, o);
    if ((lane & (kW - 1)) >= (uint32_t)o) in += n;
  }
  __syncthreads();
  if (tid < N * kW) {
    wsum[tid] = in - x;
    if ((tid & (kW - 1)) == kW - 1) wsum[N * kW + tid / kW] = in;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N; ++q) {
    v[q] = wsum[q * kW + wv] + inc[q] - v[q];
    tot[q] = wsum[N * kW + q];
  }
}

// Width class of an expert's tile of r tokens (r > 0): the narrowest whose columns hold them; tpg
// tokens fill one column tile.
__device__ __forceinline__ uint32_t tile_cls(uint32_t r, uint32_t tpg) {
  uint32_t k = 0;
#pragma unroll
  for (int q = 1; q < kNCls; ++q)
    if (r <= (uint32_t)kClsCT[q] * tpg) k = q;
  return k;
}
// An expert's c slots in tiles of tt tokens (the capacity of class k0, the batch's widest): how many
// tiles of class k it has.
__device__ __forceinline__ uint32_t n_cls_of(uint32_t c, uint32_t tt, uint32_t tpg, uint32_t k0, uint32_t k) {
  const uint32_t r = c % tt;
  return (k == k0 ? c / tt : 0u) + (r != 0u && tile_cls(r, tpg) == k ? 1u : 0u);
}
// A class runs in rounds of a tile's row blocks over the grid (the tiles dealt to the 8 XCDs in turn), so a
// few tiles past a whole round cost a round in which most of the device idles, and a class with any
// tile costs its launch's start (kClsStart more than an empty launch). kClsCost: a round of a class (256
// items; the light class's two halves of 512), by kernel trace at 1 to 8 rounds: gate/up with two terms
// 47, 34, 26 and 21 us, with three 49, 36, 26.5 and 21, down 25, 18.5, 13.4 and 11 (hidden 4096, inter
// 2048); at 2048 and 1024 27, 20, 15 and 12, and 28, 21, 15 and 12, and down 19, 15, 11.5 and 8.7: the
// same ratios within a seventh. A launch's first round takes 8 to 10 us more, an empty launch 2 to 5.
constexpr uint32_t kClsCost[kNCls] = {49, 36, 26, 21}, kClsStart = 5;
// How a GEMM's tiles meet the device: row blocks of a tile, workgroups of a launch at most (and its
// reciprocal), a light round's cost (0: the light class is not launched, see light_cost).
struct ClsGrid {
  uint32_t nrb, grid;
  float inv;
  uint32_t light;
};
// (all 16 waves of a plan compute these, where an integer division is some 35 instructions: by the
// reciprocal, corrected; the items of a batch are below 2^23, see the B rows' limit)
__device__ __forceinline__ uint32_t cls_rounds(uint32_t tiles, const ClsGrid& g) {
  const uint32_t x = (tiles + 7u) / 8u * 8u * g.nrb + g.grid - 1u;
  const uint32_t q = (uint32_t)((float)x * g.inv), r = x - q * g.grid;  // (q within one of x / grid)
  return (int32_t)r < 0 ? q - 1u : r >= g.grid ? q + 1u : q;
}
// The wide tiles that are split into a class 1 and a class 2 tile each (12 column tiles = 8 + 4): 194 wide
// gate/up tiles over 256 workgroups took 13 rounds for 12.1 rounds' work. They are split where the
// round saved is worth more than those that the narrower classes grow by.
__device__ __forceinline__ uint32_t split_wide(const uint32_t (&n)[kNCls], const ClsGrid& g, uint32_t room) {
  static_assert(kClsCT[0] == kClsCT[1] + kClsCT[2], "a wide tile is one of each");
  auto rounds = [&](uint32_t t) { return cls_rounds(t, g); };
  const uint32_t r = rounds(n[0]);
  if (r == 0) return 0u;
  const uint32_t left = n[0] - min(n[0], (r - 1u) * g.grid / g.nrb / 8u * 8u);
  if (left > room) return 0u;
  const uint32_t more =
      (rounds(n[1] + left) - rounds(n[1])) * kClsCost[1] + (rounds(n[2] + left) - rounds(n[2])) * kClsCost[2];
  return more < kClsCost[0] ? left : 0u;
}
// Whether the light tiles run in the class before them (n2 tiles) instead: where the rounds they add there
// cost less than theirs here, as with the few experts of a small layer, whose tiles of both classes
// fill a round together (8 experts, two of them a token, 64 tokens: the layer 83 us with two launches a
// GEMM, 61 with one). With two workgroups a CU the light class has no whole rounds past the first two
// halves: 94 narrow and light tiles by 16 row blocks 154 us in one launch, 30 + 115 in two. A light round
// costs less of a narrow one's where K is 1024 (down, 2 + 62 tiles by 16 row blocks: 44 + 5 us for one launch
// and an empty one, 11 + 34 for two).
constexpr uint32_t kLightShort = 18, kMergeGain = 4;
__device__ __forceinline__ bool merge_light(uint32_t n2, uint32_t n3, const ClsGrid& g) {
  if (n2 == 0u || n3 == 0u) return false;
  auto cost2 = [&](uint32_t n) { return g.grid * (cls_rounds(n, g) * kClsCost[2] + kClsStart); };
  const uint32_t items = (n3 + 7u) / 8u * 8u * g.nrb;
  const uint32_t full = items <= g.grid ? g.grid : items <= 2u * g.grid ? 2u * g.grid : items;
  return cost2(n2 + n3) + g.grid * kMergeGain <= cost2(n2) + full * g.light + g.grid * kClsStart;
}
// One GEMM's tiles: class k's n[k] tiles from tiles[base[k]]; the wide ones from index keep on are split,
// their parts following the other tiles of classes 1 and 2; the light tiles follow class 2's, to which
// they belong if merged (cls[k]: what class k runs).
struct TileSet {
  uint32_t base[kNCls], n[kNCls], keep, cls[kNCls];
};
__device__ __forceinline__ TileSet tile_set(const uint32_t* tot, uint32_t k0, const ClsGrid& g, uint32_t max_tiles) {
  TileSet t;
  uint32_t need = 0;
#pragma unroll
  for (int k = 0; k < kNCls; ++k) {
    t.n[k] = tot[k];
    need += tot[k];
  }
  const uint32_t split = k0 == 0 && need <= max_tiles ? split_wide(t.n, g, max_tiles - need) : 0u;
  t.keep = t.n[0] - split;
  t.base[0] = 0;
  t.base[1] = t.keep;
  t.base[2] = t.base[1] + t.n[1] + split;
#pragma unroll
  for (int k = 3; k < kNCls; ++k) t.base[k] = t.base[k - 1] + t.n[k - 1] + (k == 3 ? split : 0u);
#pragma unroll
  for (int k = 0; k < kNCls; ++k) t.cls[k] = k == 0 ? t.keep : t.n[k] + (k <= 2 ? split : 0u);
  static_assert(kNCls == 4, "the light class is the one after class 2");
  if (k0 <= 2 && (g.light == 0u || merge_light(t.cls[2], t.cls[3], g))) {
    t.cls[2] += t.cls[3];
    t.cls[3] = 0u;
  }
  return t;
}
// Writes the tiles of one expert (slots b0 .. b0 + c - 1), whose first of class k is the class's at[k]-th:
// the full ones of class k0, the partial one of its class (past the full ones where that is k0).
__device__ __forceinline__ void put_tiles(Tile* tiles, const TileSet& t, uint32_t e, uint32_t b0, uint32_t c, uint32_t tt,
                                          uint32_t tpg, uint32_t k0, const uint32_t* at) {
  const uint32_t full = c / tt, r = c % tt, kr = r ? tile_cls(r, tpg) : kNCls;
  auto put = [&](int k, uint32_t i, uint32_t s0, uint32_t n) {
    if (k == 0 && i >= t.keep) {
      const uint32_t d = i - t.keep, n1 = (uint32_t)kClsCT[1] * tpg;  // (a wide tile has more tokens than that)
      tiles[t.base[1] + t.n[1] + d] = Tile{e, s0, n1};
      tiles[t.base[2] + t.n[2] + d] = Tile{e, s0 + n1, n - n1};
    } else {
      tiles[t.base[k] + i] = Tile{e, s0, n};
    }
  };
#pragma unroll
  for (int k = 0; k < kNCls; ++k) {
    if ((uint32_t)k == k0)
      for (uint32_t i = 0; i < full; ++i) put(k, at[k] + i, b0 + i * tt, tt);
    if ((uint32_t)k == kr) put(k, at[k] + ((uint32_t)k == k0 ? full : 0u), b0 + full * tt, r);
  }
}

// The plan of one workgroup of kPlanThreads threads: thread e < n_experts holds expert e's count c
// (and, with own_slots, the first slot b0 its caller chose; else the slots follow in expert order).
// Slot and tile offsets by one exclusive scan (expert order) of the count and the tiles of each width
// class of both GEMMs, whose widest classes are k01 and k02; writes the tiles, the header and returns
// the expert's first slot.
struct PlanOut {
  GroupedHdr* hdr;
  Tile* tiles1;
  Tile* tiles2;
  uint32_t max_tiles1, max_tiles2;
  ClsGrid g1, g2;
};
constexpr uint32_t kPlanSums = (1 + 2 * kNCls) * (kPlanThreads / 64 + 1);
__device__ __forceinline__ uint32_t plan_tiles(uint32_t c, uint32_t b0, bool own_slots, uint32_t n_slots_in,
                                               uint32_t n_experts, uint32_t k01, uint32_t k02, uint32_t tx,
                                               uint32_t* wsum, const PlanOut& o) {
  const uint32_t tid = threadIdx.x;
  // tokens per column tile, and per tile of each GEMM's widest class
  const uint32_t tpg1 = 16u / tx, tpg2 = 16u / 3u;
  const uint32_t tt1 = cls_ct(k01) * tpg1, tt2 = cls_ct(k02) * tpg2;
  constexpr int NV = 1 + 2 * kNCls;
  uint32_t v[NV], tot[NV];
  v[0] = c;
#pragma unroll
  for (int k = 0; k < kNCls; ++k) {
    v[1 + k] = n_cls_of(c, tt1, tpg1, k01, k);
    v[1 + kNCls + k] = n_cls_of(c, tt2, tpg2, k02, k);
  }
  plan_scan<NV>(v, wsum, tot);
  if (!own_slots) b0 = v[0];
  uint32_t need1 = 0, need2 = 0;
#pragma unroll
  for (int k = 0; k < kNCls; ++k) { need1 += tot[1 + k]; need2 += tot[1 + kNCls + k]; }
  // a caller's overlapping ranges could ask for more tiles than the workspace holds: then no tile
  const bool fits = need1 <= o.max_tiles1 && need2 <= o.max_tiles2;
  const TileSet t1 = tile_set(tot + 1, k01, o.g1, o.max_tiles1);
  const TileSet t2 = tile_set(tot + 1 + kNCls, k02, o.g2, o.max_tiles2);
  if (fits && tid < n_experts) {
    put_tiles(o.tiles1, t1, tid, b0, c, tt1, tpg1, k01, v + 1);
    put_tiles(o.tiles2, t2, tid, b0, c, tt2, tpg2, k02, v + 1 + kNCls);
  }
  if (tid == 0) {
    o.hdr->n_slots = own_slots ? n_slots_in : tot[0];
#pragma unroll
    for (int k = 0; k < kNCls; ++k) {
      o.hdr->n_cls[0][k] = fits ? t1.cls[k] : 0u;
      o.hdr->n_cls[1][k] = fits ? t2.cls[k] : 0u;
    }
    o.hdr->tx = tx;
    o.hdr->bad = fits ? 0u : 1u;
  }
  return b0;
}

// start_in: a caller's slot list, expert e owning slots [start_in[e], start_in[e+1]) of n_slots_in
// (each bound clamped to n_slots_in; a range that runs backwards is empty); null: the routes'
// counts per chunk (grouped_hist_kernel), replaced by each chunk's first slot of each expert.
__global__ void __launch_bounds__(kPlanThreads) grouped_plan_kernel(
    uint32_t* __restrict__ hist, uint32_t n_chunks, uint32_t n_experts, uint32_t k01, uint32_t k02, uint32_t tx,
    const uint32_t* __restrict__ start_in, uint32_t n_slots_in, PlanOut o) {
  static_assert(AFFX_MAX_EXPERTS <= kPlanThreads, "one thread per expert in the scan");
  __shared__ uint32_t wsum[kPlanSums];
  const uint32_t tid = threadIdx.x;
  const bool own = start_in != nullptr, mine = tid < n_experts;
  uint32_t c = 0, b0 = 0;
  // (chunks eight at a time: their loads are in flight together)
  constexpr uint32_t kB = 8;
  uint32_t cb[kB];
  auto chunks = [&](uint32_t b) {
#pragma unroll
    for (uint32_t i = 0; i < kB; ++i) cb[i] = mine && b + i < n_chunks ? hist[(uint64_t)(b + i) * n_experts + tid] : 0u;
  };
  if (own) {
    if (mine) {
      const uint32_t a = min(start_in[tid], n_slots_in), e = min(start_in[tid + 1], n_slots_in);
      c = e > a ? e - a : 0u;
      b0 = a;
    }
  } else {
    for (uint32_t b = 0; b < n_chunks; b += kB) {
      chunks(b);
#pragma unroll
      for (uint32_t i = 0; i < kB; ++i) c += cb[i];
    }
  }
  uint32_t at = plan_tiles(c, b0, own, n_slots_in, n_experts, k01, k02, tx, wsum, o);
  if (own) return;
  // each chunk's first slot of this expert: its offset plus the counts of the chunks before
  for (uint32_t b = 0; b < n_chunks; b += kB) {
    if (n_chunks > kB) chunks(b);  // (else they are still here)
#pragma unroll
    for (uint32_t i = 0; i < kB; ++i)
      if (mine && b + i < n_chunks) {
        hist[(uint64_t)(b + i) * n_experts + tid] = at;
        at += cb[i];
      }
  }
}

// The whole plan of a small batch's routes in one workgroup: counts, plan and placement (see
// grouped_hist_kernel and grouped_place_kernel for what it writes and the slot order). The pairs
// are taken in groups of 64, a wave each.
constexpr uint32_t kSmallPairs = 4096;
__global__ void __launch_bounds__(kPlanThreads) grouped_plan_small_kernel(
    const uint32_t* __restrict__ sel, const float* __restrict__ w, uint32_t n_pairs, uint32_t n_tok, uint32_t top_k,
    uint32_t n_experts, uint32_t k01, uint32_t k02, uint32_t tx, const int32_t* __restrict__ tok_sigma,
    uint32_t* __restrict__ slot_tok, float* __restrict__ slot_w, int32_t* __restrict__ slot_sigma,
    uint32_t* __restrict__ ord, uint32_t* __restrict__ run, PlanOut o) {
  static_assert(AFFX_MAX_EXPERTS <= 512, "expert ids ranked by 9 ballots");
  constexpr uint32_t kW = kPlanThreads / 64, kR = kSmallPairs / kPlanThreads, kG = kSmallPairs / 64;
  __shared__ uint32_t wsum[kPlanSums];
  __shared__ uint16_t grp[kG][AFFX_MAX_EXPERTS];  // a group's count of each expert, then its first rank
  __shared__ uint32_t off[AFFX_MAX_EXPERTS];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t ng = (n_pairs + 63u) / 64u;
  uint32_t ev[kR], rank[kR];
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = r * kPlanThreads + tid;
    ev[r] = i < n_pairs ? sel[i] : ~0u;
  }
  for (uint32_t q = tid; q < ng * (AFFX_MAX_EXPERTS / 2); q += kPlanThreads) reinterpret_cast<uint32_t*>(&grp[0][0])[q] = 0u;
  for (uint32_t i = tid; i <= n_tok; i += kPlanThreads) run[i] = i * top_k;
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t g = r * kW + wv;
    rank[r] = 0;
    if (g >= ng) continue;  // (whole waves)
    const bool ok = ev[r] < n_experts;
    const uint64_t m = same_key_lanes<9>(ok ? ev[r] : 0u, ok);
    rank[r] = (uint32_t)__popcll(m & below);
    if (ok && (uint32_t)__builtin_ctzll(m) == lane) grp[g][ev[r]] = (uint16_t)__popcll(m);
  }
  __syncthreads();
  uint32_t c = 0;
  if (tid < n_experts) {
#pragma unroll 8
    for (uint32_t g = 0; g < ng; ++g) {
      const uint32_t x = grp[g][tid];
      grp[g][tid] = (uint16_t)c;
      c += x;
    }
  }
  const uint32_t b0 = plan_tiles(c, 0u, false, 0u, n_experts, k01, k02, tx, wsum, o);
  if (tid < n_experts) off[tid] = b0;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kR; ++r) {
    const uint32_t i = r * kPlanThreads + tid;
    if (i >= n_pairs) continue;
    if (!(ev[r] < n_experts)) {
      ord[i] = ~0u;
      continue;
    }
    const uint32_t pos = off[ev[r]] + grp[r * kW + wv][ev[r]] + rank[r], t = i / top_k;
    slot_tok[pos] = t;
    slot_w[pos] = w[i];
    slot_sigma[pos] = tok_sigma[t];
    ord[i] = pos;
  }
}

// The routes form's placement, in two passes over chunks of kPlaceChunk routes (four rounds of
// 256): grouped_hist_kernel counts each expert's routes per chunk, grouped_plan_kernel turns the
// counts into each chunk's first slot per expert, grouped_place_kernel gives every route its slot.
// A route's slot is its expert's offset plus the number of that expert's routes before it, so
// each expert's slots hold its routes in route order, whatever the grid.
constexpr uint32_t kPlaceChunk = 1024;

// Counts of chunk blockIdx.x into hist[chunk][expert]. Also the routes form's ord/run for the
// indices it covers: token t owns entries t k .. t k + k - 1 of ord, in route order (run[t] = t k);
// a route that names no expert of the layer keeps ~0u there (the consumers skip slot numbers past
// the slot count), grouped_place_kernel writes the slot of every other.
__global__ void __launch_bounds__(256) grouped_hist_kernel(const uint32_t* __restrict__ sel, uint32_t n_pairs,
                                                           uint32_t n_tok, uint32_t top_k, uint32_t n_experts,
                                                           uint32_t* __restrict__ hist, uint32_t* __restrict__ run,
                                                           uint32_t* __restrict__ ord) {
  __shared__ uint32_t cnt[AFFX_MAX_EXPERTS];
  const uint32_t b = blockIdx.x, tid = threadIdx.x;
  for (uint32_t e = tid; e < n_experts; e += 256) cnt[e] = 0u;
  __syncthreads();
  uint32_t ev[kPlaceChunk / 256];
#pragma unroll
  for (uint32_t r = 0; r < kPlaceChunk / 256; ++r) {
    const uint32_t i = b * kPlaceChunk + r * 256u + tid;
    ev[r] = i < n_pairs ? sel[i] : ~0u;
  }
#pragma unroll
  for (uint32_t r = 0; r < kPlaceChunk / 256; ++r) {
    const uint32_t i = b * kPlaceChunk + r * 256u + tid;
    if (ev[r] < n_experts)
      atomicAdd(&cnt[ev[r]], 1u);
    else if (i < n_pairs)
      ord[i] = ~0u;
    if (i <= n_tok) run[i] = i * top_k;
  }
  __syncthreads();
  for (uint32_t e = tid; e < n_experts; e += 256) hist[(uint64_t)b * n_experts + e] = cnt[e];
}

// The slots of chunk blockIdx.x. first[chunk][expert] is the chunk's first slot of each expert
// (grouped_plan_kernel). Routes i = chunk start + 256 r + 64 w + lane: within a wave, the lanes of
// the same expert are ranked by one ballot per expert-id bit; the (round, wave) groups are ranked
// by an exclusive scan of their per-expert counts in LDS.
__global__ void __launch_bounds__(256) grouped_place_kernel(const uint32_t* __restrict__ sel,
                                                            const float* __restrict__ w, uint32_t n_pairs,
                                                            uint32_t top_k, uint32_t n_experts,
                                                            const uint32_t* __restrict__ first,
                                                            const int32_t* __restrict__ tok_sigma,
                                                            uint32_t* __restrict__ slot_tok,
                                                            float* __restrict__ slot_w,
                                                            int32_t* __restrict__ slot_sigma,
                                                            uint32_t* __restrict__ ord) {
  static_assert(AFFX_MAX_EXPERTS <= 512, "expert ids ranked by 9 ballots");
  constexpr uint32_t NR = kPlaceChunk / 256, NG = NR * 4;  // rounds, (round, wave) groups
  __shared__ uint32_t grp[NG][AFFX_MAX_EXPERTS];
  const uint32_t b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (uint32_t q = tid; q < NG * AFFX_MAX_EXPERTS; q += 256) (&grp[0][0])[q] = 0u;
  uint32_t ev[NR], rank[NR];
#pragma unroll
  for (uint32_t r = 0; r < NR; ++r) {
    const uint32_t i = b * kPlaceChunk + r * 256u + tid;
    ev[r] = i < n_pairs ? sel[i] : ~0u;
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (uint32_t r = 0; r < NR; ++r) {
    const bool ok = ev[r] < n_experts;
    const uint64_t m = same_key_lanes<9>(ok ? ev[r] : 0u, ok);
    rank[r] = (uint32_t)__popcll(m & below);
    if (ok && (uint32_t)__builtin_ctzll(m) == lane) grp[r * 4u + wv][ev[r]] = (uint32_t)__popcll(m);
  }
  __syncthreads();
  for (uint32_t e = tid; e < n_experts; e += 256) {
    uint32_t at = 0;
#pragma unroll
    for (uint32_t g = 0; g < NG; ++g) {
      const uint32_t c = grp[g][e];
      grp[g][e] = at;
      at += c;
    }
  }
  __syncthreads();
  const uint32_t* fb = first + (uint64_t)b * n_experts;
#pragma unroll
  for (uint32_t r = 0; r < NR; ++r) {
    if (!(ev[r] < n_experts)) continue;
    const uint32_t i = b * kPlaceChunk + r * 256u + tid;
    const uint32_t pos = fb[ev[r]] + grp[r * 4u + wv][ev[r]] + rank[r];
    const uint32_t t = i / top_k;
    slot_tok[pos] = t;
    slot_w[pos] = w[i];
    slot_sigma[pos] = tok_sigma[t];
    ord[i] = pos;
  }
}

// ------------------------------------------------------------------------------------------------
// activation terms: per token an exponent and tx E4M3 terms of every element, in step order
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) grouped_prep_x_kernel(const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ xlo,
                                                             uint32_t hidden, uint32_t tx,
                                                             const uint32_t* __restrict__ ord,
                                                             const uint32_t* __restrict__ run,
                                                             uint32_t n_slots,
                                                             int32_t* __restrict__ slot_sigma,
                                                             int32_t* __restrict__ tok_sigma,
                                                             uint8_t* __restrict__ xq,
                                                             uint32_t* __restrict__ zeros,
                                                             uint32_t zero_words) {
  const uint32_t t = blockIdx.x, tid = threadIdx.x;
  if (t == 0)  // the B row of unused columns
    for (uint32_t i = tid; i < zero_words; i += 256) zeros[i] = 0u;
  __shared__ float red[4];
  const int sigma = row_terms<true>(x + (uint64_t)t * hidden, xlo ? xlo + (uint64_t)t * hidden : nullptr, hidden,
                                    tx, xq + (uint64_t)t * tx * hidden, red);
  // the exponent, for the gate/up epilogue: of the token (the routes form, whose placement hands it to
  // the slots), or to each of the token's slots (a caller's slot list)
  if (!ord) {
    if (tid == 0) tok_sigma[t] = sigma;
    return;
  }
  const uint32_t r1 = min(run[t + 1], n_slots);
  for (uint32_t i = min(run[t], r1) + tid; i < r1; i += 256) {
    const uint32_t sl = ord[i];
    if (sl < n_slots) slot_sigma[sl] = sigma;
  }
}

// ------------------------------------------------------------------------------------------------
// grouped GEMM: one workgroup = one (expert, token tile) x one row block
// ------------------------------------------------------------------------------------------------
// 8 waves, two per SIMD: on gfx950 one wave's VALU work does not overlap its own MFMAs, but it
// does overlap the other wave's. A wave owns 32 weight rows (two 16-row tiles: gate/up = one gate
// tile and the same rows of up, down = two tiles) against all 192 B columns of the tile (12 MFMA
// column tiles; a token is TX adjacent columns, 16 / TX tokens per column tile). Per MFMA step
// (128 of K):
//   - each wave decodes its own rows' A fragments in registers: one codebook lookup per quad
//     code, reused by 12 MFMAs. The table holds each codebook dword and its half-rotated form
//     (the rotation field of a block selects the table), so a code costs two VALU ops for its
//     address and one for sign and scale. Two interleaved copies (lane parity): on this kernel
//     the VALU, not the LDS bank conflicts, sets the pace, and fewer copies measured as fast as
//     four or eight;
//   - B (192 columns x 128 bytes) sits in LDS, written by direct global->LDS loads two steps at
//     a time, two steps ahead (two buffers of two steps, one workgroup barrier per two), read by all
//     eight waves; 16-byte chunks are swizzled by column so that
//     the fragment reads of 16 lanes hit 16 distinct bank groups;
//   - the packed weights of the next 1024 columns stream into a register ring, each chunk
//     reloaded as soon as the lookups of the current 1024 columns are past it.
constexpr int kGW = 8;                      // waves per workgroup (two per SIMD)
constexpr int kGRT = 16 / kGW;              // 16-row tiles per wave (a workgroup covers 256 rows)
constexpr int kGT = kGW * 64;
constexpr int kGKC = 2;                     // codebook copies (pre-rotated tables)
constexpr int kGCT = kClsCT[0];             // 16-column tiles of B per wave (a wide tile)
// A tile of CT column tiles (one of kClsCT): its B columns, the bytes of one MFMA step of B, the
// steps that one of the two B buffers holds, and a wave's direct-load instructions per buffer (8
// columns of one step each).
// Light tiles (CT = 2: at most 16 tokens of two terms, 10 of three), most tiles of a batch of a few
// hundred tokens over 256 experts, are bound by the weights' stream and the latency around it, so
// they run two workgroups a CU (at most 128 registers, 67 KB of LDS) instead of the four column
// tiles' one at 165: 111 experts of one or two tokens, gate/up 196 -> 146 us (4.6 TB/s), down
// 105 -> 79 us (hidden 4096, inter 2048; kernel trace). Per step: the products first, so that
// the next A fragments take the registers of these; block signs and scales from the fields, not the
// LDS table (the LDS is the busier: 1 %); the second column tile's products are passed over where
// the tile has no token there (an instantiation of its own for one column tile took two more
// launches and as long); four steps a buffer, so that each wave has two loads a buffer and the
// weights have four steps to arrive (a barrier waits for the loads before it). Three column tiles
// in this form (two registers spilled) measured the same as two, four spill 40.
template <int CT>
struct GTile {
  static constexpr bool kLight = CT < 4;
  static constexpr int kCols = CT * 16;
  static constexpr uint32_t kStep = kCols * 128;
  static constexpr int kNSB = kLight ? 4 : 2;
  static constexpr uint32_t kBuf = kNSB * kStep;
  static constexpr int kDma = kNSB * kCols / 8 / kGW;
};

struct GemmArgs {
  const uint8_t* base;
  uint64_t stride;
  uint64_t off[9];
  uint32_t hidden, inter;
  const uint32_t* codebook;
  const GroupedHdr* hdr;
  const Tile* tiles;
  uint32_t max_tiles;       // entries of tiles (allocated; the header says how many are used)
  const uint32_t* slot_tok;
  uint32_t n_sl;              // entries of slot_tok and slot_sigma
  uint32_t n_tok;             // tokens of the batch (a slot's token id is clamped below it)
  const int32_t* slot_sigma;  // activation exponent of the slot's token
  const uint8_t* ws;        // B rows and the zero row, addressed by 32-bit offsets from here
  uint64_t b_off, zero_off;
  uint8_t* aq;              // gate/up output [slot][3][inter], step order
  float* z;                 // down output [slot][hidden]
  float limit;
  int32_t sigma_a;
};


constexpr int kNT = 2;  // cache policy of streamed weights: non-temporal

// One unit in full (fields first, then the code chunks in order): tile t of the code and field
// planes cr, fr.
__device__ __forceinline__ void load_unit_buf(Unit& u, __amdgpu_buffer_rsrc_t cr, __amdgpu_buffer_rsrc_t fr,
                                              uint32_t t, uint32_t lane) {
#pragma unroll
  for (int q = 0; q < 3; ++q)
    u.f[q] = __builtin_amdgcn_raw_buffer_load_b32(fr, lane * 12u, t * kTileFieldBytes + 4u * q, kNT);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(cr, lane * 16u, t * kTileCodeBytes + 1024u * j, kNT);
    u.c[4 * j] = v[0]; u.c[4 * j + 1] = v[1]; u.c[4 * j + 2] = v[2]; u.c[4 * j + 3] = v[3];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Registers of a unit that the ring reloads at step M (for the next 1024 columns). Step M's
// reloads come before its table reads (those of step M + 1), so a register is reloaded at the
// first step after the last step whose table reads use it: code chunk j = c[4j..4j+3] (chunk 0
// at step 1, 1 at 3, 2 at 4, 3 at 6, 4 at 7) and field dword q (f0 at 2, f1 at 5, f2 at 7). One
// load instruction each: steps 1-6 issue one per unit, step 7 two, step 0 none.
template <int M>
__device__ __forceinline__ void ring_load(Unit& u, __amdgpu_buffer_rsrc_t cr, __amdgpu_buffer_rsrc_t fr, uint32_t t,
                                          uint32_t lane) {
  auto chunk = [&](int j) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(cr, lane * 16u, t * kTileCodeBytes + 1024u * j, kNT);
    u.c[4 * j] = v[0]; u.c[4 * j + 1] = v[1]; u.c[4 * j + 2] = v[2]; u.c[4 * j + 3] = v[3];
  };
  auto field = [&](int q) {
    u.f[q] = __builtin_amdgcn_raw_buffer_load_b32(fr, lane * 12u, t * kTileFieldBytes + 4u * q, kNT);
  };
  if constexpr (M == 1) chunk(0);
  if constexpr (M == 2) field(0);
  if constexpr (M == 3) chunk(1);
  if constexpr (M == 4) chunk(2);
  if constexpr (M == 5) field(1);
  if constexpr (M == 6) chunk(3);
  if constexpr (M == 7) { chunk(4); field(2); }
}

template <int PH, int TX, int CT>
__global__ void __launch_bounds__(kGT, GTile<CT>::kLight ? 4 : 1) grouped_gemm_kernel(GemmArgs A) {
  constexpr int TPG = 16 / TX;  // tokens per 16-column tile
  constexpr int kHalf = kGRT / 2;  // gate/up: units [0, kHalf) gate, [kHalf, kGRT) the same rows of up
  // Persistent: workgroup b runs the items (row block, token tile) w = b, b + G, b + 2G, ... (G =
  // gridDim.x, a multiple of 8). XCD-aware order: the device hands consecutive workgroups to its
  // 8 XCDs in turn, so workgroup b runs on XCD b % 8 = w % 8 for all of its items. All row blocks
  // of one token tile go to the same XCD (its L2 then holds the tile's activations for all of
  // them), consecutive tiles to different XCDs. Items are in increasing tile order per workgroup,
  // so the first item past the last tile ends the workgroup.
  const uint32_t nrb = PH == 0 ? A.inter / 128u : A.hidden / 256u;  // row blocks
  auto item_of = [&](uint32_t w, uint32_t& rb_, uint32_t& tile_) {
    const uint32_t l = w >> 3;
    rb_ = l % nrb;
    tile_ = (l / nrb) * 8u + (w & 7u);
  };
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t K = PH == 0 ? A.hidden : A.inter;
  const uint32_t nst = K / kTileCols;
  const uint32_t nsteps = nst * 8u;
  // Set-up of the first item in three memory round trips: (1) the codebook, the tile count and
  // the tiles of the first two items (read before it is known to be in use: any index below
  // max_tiles is allocated); (2) the B row of every column, then the first weights; (3) the
  // first two steps of B. Later items find their tile and B rows staged in LDS (see ep_sig), and
  // their first weights and B steps are loaded during the previous item's last 1024 columns (see
  // cont).
  constexpr int kPer = 2048 / kGT;
  uint32_t cbv[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) cbv[i] = A.codebook[tid + (uint32_t)kGT * i];
  // this instantiation's tiles: those of its width class, stored after the wider classes' tiles
  const uint32_t* ncls = A.hdr->n_cls[PH];
  uint32_t n_tiles = 0, first = 0;
#pragma unroll
  for (int k = 0; k < kNCls; ++k) {
    if (kClsCT[k] > CT) first += ncls[k];
    if (kClsCT[k] == CT) n_tiles = ncls[k];
  }
  // (entries below max_t are allocated: read before it is known whether a tile is in use)
  const uint32_t room = A.max_tiles - min(first, A.max_tiles);
  const Tile* tiles = room ? A.tiles + first : A.tiles;
  const uint32_t max_t = room ? room : 1u;
  uint32_t w = blockIdx.x, rb, tile_id, rbn, tile_n;
  item_of(w, rb, tile_id);
  item_of(w + gridDim.x, rbn, tile_n);
  Tile tl = tiles[tile_id < max_t ? tile_id : 0u];
  Tile tln = tiles[tile_n < max_t ? tile_n : 0u];  // the next item's tile
  if (tile_id >= n_tiles || tl.n == 0) return;  // (a tile in use has n >= 1: the test only makes
                                                // the loads precede the branch, in one round trip)
  bool has_next = tile_n < n_tiles && tln.n != 0;

  __shared__ __align__(16) uint32_t lut_s[Lut<kGKC, true>::kDwords];
  __shared__ __align__(16) uint2 blk_s[16];
  const uint8_t* btbl = reinterpret_cast<const uint8_t*>(blk_s);
  // B of step t in buffer (t / kNSB) % 2, written kNSB steps at a time, as many steps ahead (separate
  // arrays: the compiler can then tell the buffer being read from the one being written)
  constexpr int NSB = GTile<CT>::kNSB;
  __shared__ __align__(16) uint8_t buf0[GTile<CT>::kBuf];
  __shared__ __align__(16) uint8_t buf1[GTile<CT>::kBuf];
  uint8_t* const buf1h = buf1 + GTile<CT>::kBuf / 2;
  uint32_t* rowoff = reinterpret_cast<uint32_t*>(buf1h);  // set-up only, before buffer 1 is written
  __shared__ __align__(16) uint32_t rowoff_n[GTile<CT>::kCols];  // the next tile's, during the last 1024 columns
  // Staged at the start of each item by direct-to-LDS loads, so that neither the epilogue nor the
  // step to the next item waits for memory: the item's activation exponents (gate/up: one per
  // slot of the tile, 128 entries) and row scales (256 bf16: the 128 gate and 128 up rows, or the
  // 256 down rows), the next item's B rows (gate/up: its slots' tokens) and the tile of the item
  // after it.
  __shared__ __align__(16) uint32_t ep_sig[128];
  __shared__ __align__(16) uint32_t ep_rs[128];
  __shared__ __align__(16) uint32_t ep_tok[128];
  __shared__ __align__(16) uint32_t ep_tile[64];
  const uint8_t* lut = reinterpret_cast<const uint8_t*>(lut_s);

  // ---- per-item state: the expert's planes, this wave's row tiles, the B rows -----------------
  // the wave's 16-row tiles: gate/up = gate tile rt0 (unit 0) and the same rows of up (unit 1);
  // down = two consecutive tiles. Unit r's code/field planes: (c0, f0) for the gate unit or down,
  // (c1, f1) for the up unit.
  const uint64_t cbytes = (uint64_t)(PH == 0 ? A.inter : A.hidden) * code_row_bytes(K);
  const uint64_t fbytes = (uint64_t)(PH == 0 ? A.inter : A.hidden) * field_row_bytes(K);
  const uint8_t* ex;
  __amdgpu_buffer_rsrc_t c0, f0, c1, f1;
  uint32_t rt0;
  auto set_item = [&](const Tile& t, uint32_t rb_) {
    ex = A.base + (uint64_t)t.expert * A.stride;
    c0 = buffer_rsrc(ex + A.off[PH == 0 ? kGateCodes : kDownCodes], (uint32_t)cbytes);
    f0 = buffer_rsrc(ex + A.off[PH == 0 ? kGateFields : kDownFields], (uint32_t)fbytes);
    c1 = buffer_rsrc(ex + A.off[PH == 0 ? kUpCodes : kDownCodes], (uint32_t)cbytes);
    f1 = buffer_rsrc(ex + A.off[PH == 0 ? kUpFields : kDownFields], (uint32_t)fbytes);
    rt0 = PH == 0 ? rb_ * 8u + kHalf * wv : rb_ * 16u + kGRT * wv;
  };
  auto rt_of = [&](int r) -> uint32_t { return PH == 0 ? rt0 + (r % kHalf) : rt0 + r; };
  Unit u[kGRT];
  auto load_units = [&]() {
#pragma unroll
    for (int r = 0; r < kGRT; ++r)
      load_unit_buf(u[r], PH == 0 && r >= kHalf ? c1 : c0, PH == 0 && r >= kHalf ? f1 : f0, rt_of(r) * nst, lane);
  };
  // B row of column tid (threads below GTile<CT>::kCols): a column past the tile's tokens reads the tile's
  // first slot (unconditional load) and gets the zero row
  // (these and the per-item lane values below are derived from an opaque copy of the thread index
  // where they are used: derived once, outside the item loop, they were held across it, spilled,
  // and every reload from scratch memory waited for all the loads in flight)
  auto tid_now = [&]() -> uint32_t {
    uint32_t z = 0u;
    AFFX_PIN(z);  // (the lane count below is made where it is used, from nothing held across)
    return wv * 64u + __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
  };
  const uint32_t bcol_j = (tid >> 4) * TPG + (tid & 15u) / TX;
  auto brow_load = [&](const Tile& t) -> uint32_t {
    const uint32_t bslot = t.slot0 + ((tid < GTile<CT>::kCols && (tid & 15u) < TX * TPG && bcol_j < t.n) ? bcol_j : 0u);
    return PH == 0 ? min(A.slot_tok[bslot], A.n_tok - 1u) : bslot;
  };
  // the same from the tokens staged in ep_tok (slot t.slot0 + j at entry j)
  auto brow_staged = [&](const Tile& t) -> uint32_t {
    const uint32_t tp = tid_now(), bj = (tp >> 4) * TPG + (tp & 15u) / TX;
    const uint32_t j = (tp < GTile<CT>::kCols && (tp & 15u) < TX * TPG && bj < t.n) ? bj : 0u;
    return PH == 0 ? min(ep_tok[j], A.n_tok - 1u) : t.slot0 + j;
  };
  // (B rows are addressed by 32-bit offsets into the workspace, which the host checks fit, so the
  // offsets are computed in 32 bits)
  auto rowoff_store = [&](const Tile& t, uint32_t brow) {
    const uint32_t tp = tid_now(), bj = (tp >> 4) * TPG + (tp & 15u) / TX;
    const bool used = tp < GTile<CT>::kCols && (tp & 15u) < TX * TPG && bj < t.n;
    if (tp < GTile<CT>::kCols)
      rowoff[tp] = used ? (uint32_t)A.b_off + (brow * TX + (tp & 15u) % TX) * K : (uint32_t)A.zero_off;
  };
  auto rowoff_store_next = [&](const Tile& t, uint32_t brow) {
    const uint32_t tp = tid_now(), bj = (tp >> 4) * TPG + (tp & 15u) / TX;
    const bool used = tp < GTile<CT>::kCols && (tp & 15u) < TX * TPG && bj < t.n;
    if (tp < GTile<CT>::kCols)
      rowoff_n[tp] = used ? (uint32_t)A.b_off + (brow * TX + (tp & 15u) % TX) * K : (uint32_t)A.zero_off;
  };
  // DMA lane map: a wave's instruction i of a buffer writes columns 8b..8b+7 of one of its steps,
  // lane l to LDS slot l & 7 of column 8b + (l >> 3) (dma_at: b and the step; light tiles spread
  // the steps of a buffer over the waves); slot p of column col holds global chunk p ^ f(col),
  // f(col) = (c ^ (c >> 3)) & 7 with c = col & 15 (the column within its 16-column tile), that
  // is (col & 7) ^ ((col >> 3) & 1). A fragment read (lane = column c + 16 k-group) then puts lanes
  // 0-7, 8-15 (and so on) on 8 distinct 16-byte bank groups, and lanes 0-15 on 16.
  // (sized for the wide tile, a narrow one uses the first entries: with a size that depends on CT,
  // captured by the lambdas below, ROCm 7.2's hipcc emits no host stub for the kernel)
  constexpr int kPerStep = GTile<CT>::kLight ? GTile<CT>::kDma : GTile<CT>::kDma / 2;  // column groups of a wave
  auto dma_b = [&](int i) -> uint32_t {  // (i < kPerStep) column group of the wave's i-th
    return GTile<CT>::kLight ? (kPerStep * wv + (uint32_t)i) % (2u * CT) : kPerStep * wv + (uint32_t)i;
  };
  uint32_t roff[GTile<kGCT>::kDma / 2];
  auto roff_load = [&]() {
    const uint32_t lp = tid_now() & 63u;
#pragma unroll
    for (int i = 0; i < kPerStep; ++i) {
      const uint32_t col = 8u * dma_b(i) + (lp >> 3);
      const uint32_t q = (lp & 7u) ^ ((col & 7u) ^ ((col >> 3) & 1u));
      roff[i] = rowoff[col] + (q << 4);
    }
  };
  auto roff_load_next = [&]() {
    const uint32_t lp = tid_now() & 63u;
#pragma unroll
    for (int i = 0; i < kPerStep; ++i) {
      const uint32_t col = 8u * dma_b(i) + (lp >> 3);
      const uint32_t q = (lp & 7u) ^ ((col & 7u) ^ ((col >> 3) & 1u));
      roff[i] = rowoff_n[col] + (q << 4);
    }
  };
  const __amdgpu_buffer_rsrc_t wsr = buffer_rsrc(A.ws, 0xFFFFFFFFu);
  // steps t .. t + kNSB - 1 of B into buf
  auto dma = [&](uint8_t* buf, uint32_t t) {
    if constexpr (GTile<CT>::kLight) {
#pragma unroll
      for (int i = 0; i < kPerStep; ++i) {
        const uint32_t st = (kPerStep * wv + (uint32_t)i) / (2u * CT);  // the step within the buffer
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wsr, AFFX_LDS_PTR(buf + st * GTile<CT>::kStep + dma_b(i) * 1024u), 16,
                                                 roff[i], (t + st) * 128u, 0, 0);
      }
    } else {
#pragma unroll
      for (int st = 0; st < NSB; ++st)
#pragma unroll
        for (int i = 0; i < kPerStep; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wsr, AFFX_LDS_PTR(buf + st * GTile<CT>::kStep + dma_b(i) * 1024u), 16,
                                                   roff[i], (t + st) * 128u, 0, 0);
    }
  };

  // ---- set-up of the first item (B row loads first: the set-up waits for them, and loads
  // complete in issue order; then the weights; the codebook copies while they are in flight) ---
  {
    const uint32_t brow = brow_load(tl);
    __builtin_amdgcn_sched_barrier(0);
    set_item(tl, rb);
    load_units();
    __builtin_amdgcn_sched_barrier(0);
    build_lut<kGKC, kGT, kPer, true>(lut_s, cbv, tid);
    build_blk_tbl(blk_s, tid);
    rowoff_store(tl, brow);
    __syncthreads();
    roff_load();
    dma(buf0, 0);
    __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }

  // epilogue helpers: accumulator lane (c, kg), element v = D[4 kg + v][c]: row 4 kg + v of the
  // row tile, column c. (Every accumulator index is a compile-time constant: a runtime index
  // would put the whole accumulator array in scratch memory.)
  auto terms = [&](float d) -> float {
    const float d1 = row_shl<1>(d);
    if constexpr (TX == 2) {
      return d + d1 * 0.0625f;
    } else {
      const float d2 = row_shl<2>(d);
      return d + d1 * 0.0625f + d2 * 0.00390625f;
    }
  };
  auto bf16x4 = [](uint2 v, float (&o)[4]) {
    o[0] = __uint_as_float(v.x << 16);
    o[1] = __uint_as_float(v.x & 0xFFFF0000u);
    o[2] = __uint_as_float(v.y << 16);
    o[3] = __uint_as_float(v.y & 0xFFFF0000u);
  };
  const float L = A.limit;

  const __amdgpu_buffer_rsrc_t sig_r = buffer_rsrc(A.slot_sigma, 4u * A.n_sl);
  const __amdgpu_buffer_rsrc_t tok_r = buffer_rsrc(A.slot_tok, 4u * A.n_sl);
  const __amdgpu_buffer_rsrc_t tile_r = buffer_rsrc(tiles, (uint32_t)sizeof(Tile) * max_t);
  auto lds4 = [&](__amdgpu_buffer_rsrc_t r, uint32_t* dst, uint32_t byte_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, AFFX_LDS_PTR(dst), 4, (tid_now() & 63u) * 4u, byte_off, 0, 0);
  };
  for (;;) {
    // ---- staging (one wave each; issued before the steps' loads, so the steps' exact wait
    // counts are unchanged: loads complete in issue order) ----------------------------------------
    {
      uint32_t rb2s, tile2s;
      item_of(w + 2u * gridDim.x, rb2s, tile2s);
      if (wv == 0) {
        if constexpr (PH == 0) {
          lds4(sig_r, ep_sig, 4u * tl.slot0);
          lds4(sig_r, ep_sig + 64, 4u * tl.slot0 + 256u);
        }
      } else if (wv == 1) {
        const __amdgpu_buffer_rsrc_t rs_r =
            buffer_rsrc(ex + A.off[PH == 0 ? kGateRs : kDownRs], 2u * (PH == 0 ? A.inter : A.hidden));
        if constexpr (PH == 0) {
          lds4(rs_r, ep_rs, 256u * rb);
          lds4(buffer_rsrc(ex + A.off[kUpRs], 2u * A.inter), ep_rs + 64, 256u * rb);
        } else {
          lds4(rs_r, ep_rs, 512u * rb);
          lds4(rs_r, ep_rs + 64, 512u * rb + 256u);
        }
      } else if (wv == 2) {
        if constexpr (PH == 0) {
          if (has_next) {
            lds4(tok_r, ep_tok, 4u * tln.slot0);
            lds4(tok_r, ep_tok + 64, 4u * tln.slot0 + 256u);
          }
        }
      } else if (wv == 3) {
        lds4(tile_r, ep_tile, (uint32_t)sizeof(Tile) * (tile2s < max_t ? tile2s : 0u));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // this item's row tiles (set_item moves rt0 to the next item's during the last 1024 columns)
    const uint32_t rt0_cur = rt0;
    auto rt_cur = [&](int r) -> uint32_t { return PH == 0 ? rt0_cur + (r % kHalf) : rt0_cur + r; };
    // The next item's first weights stream into the register ring during this item's last 1024
    // columns, in place of the ring's idle reloads, and its first two steps of B go out at step 6
    // of those columns, so the step to the next item waits for no load (a burst of the next item's
    // loads there or before the epilogue was held by the memory pipeline). Needs the next item's B
    // rows staged (visible after the first barrier, so at least two sets of 1024 columns).
    const bool cont = has_next && nst >= 2u;
    const uint32_t n_cur = tl.n;
    // the lane's table copy, fragment offsets and epilogue position (derived per item: see tid_now)
    const uint32_t lane_p = tid_now() & 63u;
    const uint32_t copy4 = (lane_p & (kGKC - 1)) * 4u;
    const uint32_t c = lane_p & 15, kg = lane_p >> 4;
    const uint32_t bo0 = c * 128u + (((2u * kg) ^ ((c ^ (c >> 3)) & 7u)) << 4);
    const uint32_t bo1 = c * 128u + (((2u * kg + 1u) ^ ((c ^ (c >> 3)) & 7u)) << 4);
    v8i a_cur[kGRT];
#pragma unroll
    for (int r = 0; r < kGRT; ++r) {
      uint32_t raw[8], sx[4];
      lut_lookup_step<kGKC, true>(u[r], lut, btbl, copy4, 0, raw, sx);
      a_cur[r] = lut_finish(raw, sx);
    }
    uint32_t raw_c[4];  // the table reads in flight from one quarter of a step to the next (heavy tiles)
    uint2 sx_c;
    if constexpr (!GTile<CT>::kLight) lut_lookup_block<kGKC, 1, 0>(u[0], lut, btbl, copy4, raw_c, sx_c);
    v4f acc[kGRT][CT];
#pragma unroll
    for (int r = 0; r < kGRT; ++r)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[r][ct] = v4f{0.f, 0.f, 0.f, 0.f};

    // ---- main loop: 1024 columns of K per iteration, eight MFMA steps ---------------------------
    // (each step is instantiated with its index as a constant: the ring loads, the code positions
    // and the wait counts of a step are all fixed at compile time)
    auto step = [&](auto mc, uint32_t s, bool more) {
      constexpr int m = decltype(mc)::value;
      const uint8_t* bcur = ((m / NSB) % 2 ? buf1 : buf0) + (m % NSB) * GTile<CT>::kStep;
      // B of the next NSB steps, issued at the top of a buffer's first step into the other buffer
      // (read before the barrier that ended the step before): the workgroup then needs one barrier
      // per NSB steps. Past the last step the loads repeat the last steps' B into a buffer nobody
      // reads again, so the count of loads in flight is the same on every path.
      if constexpr (m % NSB == 0) {
        const uint32_t t2 = s * 8u + m + NSB;
        // (in the last 1024 columns' last buffer: the next item's first steps, which go to buffer 0
        // as the steps after these would)
        const bool nx = m == 8 - NSB && !more && cont;
        if constexpr (m == 8 - NSB) {
          if (nx) roff_load_next();
        }
        dma((m / NSB) % 2 ? buf0 : buf1, nx ? 0u : t2 < nsteps ? t2 : nsteps - NSB);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ring loads for the next 1024 columns; after the last ones, the same loads of tile 0 (hot
      // in the cache, read by every workgroup): their registers are not read again, and issuing
      // them keeps the count of loads in flight the same on every path
      if constexpr (m != 0) {
#pragma unroll
        for (int r = 0; r < kGRT; ++r)
          ring_load<m>(u[r], PH == 0 && r >= kHalf ? c1 : c0, PH == 0 && r >= kHalf ? f1 : f0,
                       more ? rt_of(r) * nst + s + 1 : cont ? rt_of(r) * nst : 0u, lane);
      }
      __builtin_amdgcn_sched_barrier(0);
      // (heavy tiles) The step is four quarters. Each looks up one block (four codes: addresses and table
      // reads) of the next step's A fragments, the last quarter the first block of the step after, and
      // finishes (sign and scale) the block that the quarter before looked up, between its share of
      // the MFMAs, whose B fragments are read two column tiles ahead: about three VALU operations an
      // MFMA all along the step. (A unit's eight codes in one of twelve groups, finished four groups
      // later, left most MFMAs without and some with fifteen: C4 2044 -> 2028 us, the same
      // process.) The VALU of one wave runs while the matrix core works through the other wave's
      // MFMAs. Few table reads and next A fragments are live at a time: with two waves per SIMD a wave
      // has 256 registers, accumulators included. (Step 0 of the next 1024 columns after step 7: the
      // ring has reloaded every register those reads use.)
      constexpr int mn = (m + 1) & 7;
      v8i a_next[kGRT];
      auto bread = [&](int ct) -> v8i {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(bcur + ct * 2048 + bo0);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(bcur + ct * 2048 + bo1);
        v8i b;
        b[0] = (int)lo[0]; b[1] = (int)lo[1]; b[2] = (int)lo[2]; b[3] = (int)lo[3];
        b[4] = (int)hi[0]; b[5] = (int)hi[1]; b[6] = (int)hi[2]; b[7] = (int)hi[3];
        return b;
      };
      if constexpr (GTile<CT>::kLight) {
        // (four waves a SIMD: the other waves' work covers the table reads' and MFMAs' latency)
        uint32_t rawn[kGRT][8], sxn[kGRT][2];
        static_for<0, CT>([&](auto cc) {
          constexpr int ct = decltype(cc)::value;
          if (ct > 0 && n_cur <= (uint32_t)(ct * TPG)) return;  // no token there (the same for the whole workgroup)
          const v8i bq = bread(ct);
#pragma unroll
          for (int r = 0; r < kGRT; ++r) acc[r][ct] = mfma(a_cur[r], bq, acc[r][ct]);
        });
        __builtin_amdgcn_sched_barrier(0);  // (the products first: their A fragments' registers are then free)
        static_for<0, kGRT>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          pin_step<mn>(u[r]);
          lut_lookup<kGKC, mn, true>(u[r], lut, btbl, copy4, rawn[r], sxn[r]);
        });
#pragma unroll
        for (int r = 0; r < kGRT; ++r) {
          a_next[r] = lut_finish(rawn[r], sxn[r]);
          AFFX_PIN(a_next[r]);
        }
      } else {
      v8i bq0 = bread(0), bq1 = bread(1);
      static_for<0, 4>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        constexpr int q = (g + 1) & 3;  // the quarter looked up: block q & 1 of unit q >> 1
        uint32_t rawl[4];
        uint2 sxl;
        lut_lookup_block<kGKC, g == 3 ? (m + 2) & 7 : mn, q & 1>(u[q >> 1], lut, btbl, copy4, rawl, sxl);
        static_for<0, CT / 4>([&](auto cc) {
          constexpr int ct = g * (CT / 4) + decltype(cc)::value;
          v8i bq2;
          if constexpr (ct + 2 < CT) bq2 = bread(ct + 2);
#pragma unroll
          for (int r = 0; r < kGRT; ++r) acc[r][ct] = mfma(a_cur[r], bq0, acc[r][ct]);
          bq0 = bq1;
          if constexpr (ct + 2 < CT) bq1 = bq2;
        });
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a_next[g >> 1][4 * (g & 1) + i] = (int)((raw_c[i] ^ sx_c.x) + sx_c.y);
          raw_c[i] = rawl[i];
        }
        sx_c = sxl;
#pragma unroll
        for (int i = 0; i < kGRT * CT / 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int r = 0; r < kGRT; ++r) AFFX_PIN(a_next[r]);  // computed here, not sunk into the next step
      }
      // the accumulators are materialised here (else the compiler sinks every MFMA below all
      // eight steps' table reads and holds those in registers). They stay in VGPRs: a kernel that
      // names no AGPR gets its whole register budget as VGPRs, where one that does is split half
      // and half, and the other half is then too small for the rest of the step.
#pragma unroll
      for (int r = 0; r < kGRT; ++r)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) AFFX_PIN(acc[r][ct]);
#pragma unroll
      for (int r = 0; r < kGRT; ++r) a_cur[r] = a_next[r];
      // After a buffer's last step t: the B of the next NSB steps (issued at the top of step t - NSB + 1)
      // is in LDS once every wave's loads up to them have landed. Loads complete in issue order, so
      // at most the loads issued after them may still be outstanding: the ring loads of the
      // buffer's steps (2 units x {0,1,1,1,1,1,1,2} by step).
      if constexpr (m % NSB == NSB - 1) {
        constexpr int c[8] = {0, 1, 1, 1, 1, 1, 1, 2};
        constexpr int k = kGRT * (NSB == 2 ? c[m - 1] + c[m] : c[m - (NSB - 1)] + c[m - (NSB - 2)] + c[m - 1] + c[m]);
        __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(k));
        __builtin_amdgcn_s_barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    for (uint32_t s = 0; s < nst; ++s) {
      const bool more = s + 1 < nst;
      if (!more && cont) {
        // the next item's planes and B-row offsets (published by the barrier of the first buffer)
        rowoff_store_next(tln, brow_staged(tln));
        set_item(tln, rbn);
      }
      step(IConst<0>{}, s, more);
      step(IConst<1>{}, s, more);
      step(IConst<2>{}, s, more);
      step(IConst<3>{}, s, more);
      step(IConst<4>{}, s, more);
      step(IConst<5>{}, s, more);
      step(IConst<6>{}, s, more);
      step(IConst<7>{}, s, more);
    }
    // every wave is past its last B read; step 7 waited for every direct-to-LDS load (the next
    // item's first B steps included), and the ring's last loads may stay in flight
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    // ---- epilogue inputs, from the staging in LDS -------------------------------------------
    // (gate/up: the activation exponent of the lane's token in each column tile, columns past the
    // tile's tokens read its last token and store nothing; the row scales. Down: row scales.)
    const bool next = has_next;
    int sig[PH == 0 ? CT : 1];
    uint2 rgw[kHalf], ruw[kHalf], rdw[kGRT];
    if constexpr (PH == 0) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const uint32_t j = ct * TPG + c / TX;
        sig[ct] = (int)ep_sig[j < tl.n ? j : tl.n - 1u];
      }
#pragma unroll
      for (int p = 0; p < kHalf; ++p) {
        const uint32_t loc = (rt_cur(p) - rb * 8u) * 16u + 4u * kg;  // row within the gate/up row block
        rgw[p] = *reinterpret_cast<const uint2*>(ep_rs + loc / 2);
        ruw[p] = *reinterpret_cast<const uint2*>(ep_rs + 64 + loc / 2);
      }
    } else {
#pragma unroll
      for (int r = 0; r < kGRT; ++r)
        rdw[r] = *reinterpret_cast<const uint2*>(ep_rs + ((rt_cur(r) - rb * 16u) * 16u + 4u * kg) / 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    // this item's tile, kept for its epilogue
    const Tile tl_cur = tl;
    uint32_t brow2 = 0;
    if (next && !cont) brow2 = brow_staged(tln);
    __builtin_amdgcn_sched_barrier(0);

    // ---- epilogue arithmetic and stores ------------------------------------------------------
    // Gate/up: the SwiGLU terms go to LDS first, term t of the tile's token j at row x of the row
    // block (x < 128) at stg(t) + j * 128 + x (terms 0-1 in the lower half of buffer 1, term 2 in its
    // upper half past the B-row offsets the next item writes there; the buffer is free once the
    // steps are done),
    // and then out in 16-byte pieces: each (token, term) is 128 bytes of the output row, four runs
    // of 32 at a 128-byte stride in the down GEMM's step order. (Written from the accumulator
    // lanes, two or four bytes per lane and term: 36 narrow stores per wave, whose
    // acknowledgements the next item then waited for.)
    constexpr uint32_t kTT = CT * TPG;  // tokens of a tile of this class
    auto stg = [&](uint32_t t) -> uint8_t* { return t < 2 ? buf1 + t * kTT * 128u : buf1h + 1024u; };
    static_assert(2u * kTT * 128u <= GTile<CT>::kBuf / 2 && 1024u + kTT * 128u <= GTile<CT>::kBuf / 2, "");
    if constexpr (PH == 0) {
      static_for<0, kHalf>([&](auto pc) {
        constexpr int p = decltype(pc)::value;
        const uint32_t row0 = rt_cur(p) * 16u + 4u * kg;
        float rg[4], ru[4];
        bf16x4(rgw[p], rg);
        bf16x4(ruw[p], ru);
        const uint32_t xloc = row0 - rb * 128u;  // the row within the row block
        static_for<0, CT>([&](auto cc) {
          constexpr int ct = decltype(cc)::value;
          if (ct * TPG >= tl_cur.n) return;  // no token in this column tile (the same for the whole wave)
          float sg[4], su[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            sg[v] = terms(acc[p][ct][v]);
            su[v] = terms(acc[p + kHalf][ct][v]);
          }
          const uint32_t j = ct * TPG + c / TX;
          if constexpr (TX == 2) {
            // the lane pair (2i, 2i + 1) shares token i's four rows: the even lane (whose
            // combined terms these are) keeps rows 0-1 and hands rows 2-3 to the odd lane, so
            // every lane runs the SwiGLU and the term split on two values
            const bool odd = (c & 1u) != 0;
            float g2[2], u2[2];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
              const float gu = row_shr<1>(sg[v + 2]), uu = row_shr<1>(su[v + 2]);
              g2[v] = odd ? gu : sg[v];
              u2[v] = odd ? uu : su[v];
            }
            if (j < tl_cur.n) {
              float a2[2];
#pragma unroll
              for (int v = 0; v < 2; ++v) {
                float gv = ldexpf(g2[v], -sig[ct]) * (odd ? rg[v + 2] : rg[v]);
                float uv = ldexpf(u2[v], -sig[ct]) * (odd ? ru[v + 2] : ru[v]);
                gv = (L < gv) ? L : gv;  // SwiGLU with the asymmetric clamp: src/engine/ops.cpp:47-60
                const float lo = (-L < uv) ? uv : -L;
                uv = (lo < L) ? lo : L;
                const float e = __builtin_amdgcn_exp2f(-gv * 1.44269504f);
                a2[v] = ldexpf(gv * __builtin_amdgcn_rcpf(1.0f + e) * uv, A.sigma_a);
              }
              uint32_t o0, o1, o2;
              split3x2(a2[0], a2[1], o0, o1, o2);
              const uint32_t at = j * 128u + xloc + (odd ? 2u : 0u);
              *reinterpret_cast<uint16_t*>(stg(0) + at) = (uint16_t)o0;
              *reinterpret_cast<uint16_t*>(stg(1) + at) = (uint16_t)o1;
              *reinterpret_cast<uint16_t*>(stg(2) + at) = (uint16_t)o2;
            }
          } else if (c % TX == 0 && c < TX * TPG && j < tl_cur.n) {
            float a[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              float gv = ldexpf(sg[v], -sig[ct]) * rg[v];
              float uv = ldexpf(su[v], -sig[ct]) * ru[v];
              gv = (L < gv) ? L : gv;  // SwiGLU with the asymmetric clamp: src/engine/ops.cpp:47-60
              const float lo = (-L < uv) ? uv : -L;
              uv = (lo < L) ? lo : L;
              // (hardware exp2 and reciprocal: a few ulp, far inside the path's tolerance, against
              // some thirty VALU ops per element for expf and an IEEE division; gv -> -inf gives
              // exp -> inf, reciprocal 0, a signed zero)
              const float e = __builtin_amdgcn_exp2f(-gv * 1.44269504f);
              a[v] = ldexpf(gv * __builtin_amdgcn_rcpf(1.0f + e) * uv, A.sigma_a);
            }
            uint32_t o0, o1, o2;
            split3x4(a[0], a[1], a[2], a[3], o0, o1, o2);
            const uint32_t at = j * 128u + xloc;
            *reinterpret_cast<uint32_t*>(stg(0) + at) = o0;
            *reinterpret_cast<uint32_t*>(stg(1) + at) = o1;
            *reinterpret_cast<uint32_t*>(stg(2) + at) = o2;
          }
        });
      });
      __syncthreads();
      // out: piece q (16 bytes) of (token j, term t), k = (t n + j) 8 + q
      const uint32_t n = tl_cur.n, d0 = kperm(rb * 128u);
      const uint32_t tp = tid_now();
      for (uint32_t k = tp; k < n * 24u; k += kGT) {
        const uint32_t q = k & 7u, jt = k >> 3, t = jt / n, j = jt - t * n;
        const u32x4 v = *reinterpret_cast<const u32x4*>(stg(t) + j * 128u + q * 16u);
        *reinterpret_cast<u32x4*>(A.aq + ((uint64_t)(tl_cur.slot0 + j) * 3 + t) * A.inter + d0 + (q >> 1) * 128u +
                                  (q & 1u) * 16u) = v;
      }
    } else {
      static_for<0, kGRT>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        const uint32_t row0 = rt_cur(r) * 16u + 4u * kg;
        float rd[4];
        bf16x4(rdw[r], rd);
        static_for<0, CT>([&](auto cc) {
          constexpr int ct = decltype(cc)::value;
          if (ct * TPG >= tl_cur.n) return;  // no token in this column tile (the same for the whole wave)
          float sd[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) sd[v] = terms(acc[r][ct][v]);
          const uint32_t j = ct * TPG + c / TX;
          if (c % TX == 0 && c < TX * TPG && j < tl_cur.n) {
            float4 o;
            o.x = ldexpf(sd[0], -A.sigma_a) * rd[0];
            o.y = ldexpf(sd[1], -A.sigma_a) * rd[1];
            o.z = ldexpf(sd[2], -A.sigma_a) * rd[2];
            o.w = ldexpf(sd[3], -A.sigma_a) * rd[3];
            *reinterpret_cast<float4*>(A.z + (uint64_t)(tl_cur.slot0 + j) * A.hidden + row0) = o;
          }
        });
      });
    }
    if (!next) break;

    // ---- next item's weights and first two steps of B; the tile of the item after it (staged,
    // read before the next item's staging overwrites it) -----------------------------------------
    Tile tl3;
    tl3.expert = __builtin_amdgcn_readfirstlane(ep_tile[0]);
    tl3.slot0 = __builtin_amdgcn_readfirstlane(ep_tile[1]);
    tl3.n = __builtin_amdgcn_readfirstlane(ep_tile[2]);
    if (!cont) {
      set_item(tln, rbn);
      load_units();
      rowoff_store(tln, brow2);
      __syncthreads();
      roff_load();
      dma(buf0, 0);
    }
    w += gridDim.x;
    rb = rbn;
    tl = tln;
    item_of(w + gridDim.x, rbn, tile_n);
    tln = tl3;
    has_next = tile_n < n_tiles && tln.n != 0;
    __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
}

// y[t][h] (+)= sum_i wt[ord[i]] * z[ord[i]][h] over token t's slots i = run[t] .. run[t+1]-1, in
// that order (the routes-in entry lists a token's slots in route order).
__global__ void __launch_bounds__(256) grouped_combine_kernel(const float* __restrict__ z,
                                                              const uint32_t* __restrict__ ord,
                                                              const uint32_t* __restrict__ run,
                                                              const float* __restrict__ slot_w,
                                                              uint32_t n_slots, uint32_t hidden,
                                                              float* __restrict__ y, int accumulate) {
  const uint32_t t = blockIdx.y;
  const uint32_t h = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (h >= hidden) return;
  float4 acc = accumulate ? *reinterpret_cast<const float4*>(y + (uint64_t)t * hidden + h)
                          : make_float4(0.f, 0.f, 0.f, 0.f);
  const uint32_t r1 = min(run[t + 1], n_slots);
  for (uint32_t i = min(run[t], r1); i < r1; ++i) {
    const uint32_t s = ord[i];
    if (s >= n_slots) continue;
    const float wt = slot_w[s];
    const float4 v = *reinterpret_cast<const float4*>(z + (uint64_t)s * hidden + h);
    acc.x += wt * v.x;
    acc.y += wt * v.y;
    acc.z += wt * v.z;
    acc.w += wt * v.w;
  }
  *reinterpret_cast<float4*>(y + (uint64_t)t * hidden + h) = acc;
}

}  // namespace affx

using namespace affx;

namespace {


constexpr uint32_t kSplitRoom = 64;
struct GroupedWs {
  uint64_t hdr, run, slot_tok, slot_w, ord, hist, tiles1, tiles2, sigma, tok_sigma, zeros, xq, aq, z, total;
  uint32_t max_tiles1, max_tiles2;
};

// The widest class of a batch of T tokens and P slots over E experts (a token is `terms` columns): of those
// two of whose tiles hold the batch, the one whose rounds cost least if every expert has the mean's
// tokens. An expert with more tokens than one tile is cut into more of them, each of which decodes
// its weights again; a batch this small has few such (24 tokens over 256 experts: none at uniform
// routes), so that is the narrowest, and the wider classes, whose launches would find no tile, are
// not launched (4-5 us each). Where most experts would be cut it is the narrowest only if the device has
// room for the tiles (32 tokens that all take 8 experts: 63 us in two light tiles each, 69 in one of
// four columns; all 16 experts: 100 and 79).
uint32_t widest_cls(uint32_t T, uint64_t P, uint32_t E, uint32_t terms, uint32_t nrb, uint32_t grid) {
  uint32_t k = 0;
  uint64_t least = ~0ull;
  for (int q = 0; q < kNCls; ++q) {
    const uint64_t cap = (uint64_t)kClsCT[q] * (16 / terms);
    if (q > 0 && T > 2u * cap) break;
    const uint64_t tiles = (P + E * cap - 1) / (E * cap) * E;
    const uint64_t cost = ((tiles + 7) / 8 * 8 * nrb + grid - 1) / grid * kClsCost[q];
    if (cost <= least) {
      least = cost;
      k = (uint32_t)q;
    }
  }
  return k;
}

// A light round's cost, 0 where the light tiles join the four-column ones whatever the routes: where the partial
// tiles (one an expert) fill at most two rounds, and some of them are of four columns, a class of their own
// saves at most 3 of kClsCost's units by merge_light's costs, and where the plan merges them its empty launch
// is 2 us (64 experts of 2048 x 1024, top 4, 1024 tokens: 170.4 us with it in both GEMMs, 167.1 without; 448
// shapes, none slower). A mean of four columns of tokens an expert keeps out the batches whose tiles are all
// light.
uint32_t light_cost(uint64_t P, uint32_t E, uint32_t k0, uint32_t terms, uint32_t nrb, uint32_t grid, uint32_t k) {
  const uint64_t items = (uint64_t)(E + 7u) / 8u * 8u * nrb;
  if (k0 <= 2u && items <= 2u * grid && P >= (uint64_t)E * kClsCT[2] * (16 / terms)) return 0u;
  return k > 1024 ? kClsCost[3] : kLightShort;
}

// chunks of the routes form's placement: they cover the routes and the run entries 0 .. T
uint64_t place_chunks(uint32_t T, uint64_t P) {
  const uint64_t n = P > T ? P : (uint64_t)T + 1;
  return (n + kPlaceChunk - 1) / kPlaceChunk;
}

// T tokens, room for P slots (the routes form: T * top_k)
GroupedWs grouped_ws(uint32_t T, uint64_t P, uint32_t E, uint32_t hidden, uint32_t inter, uint32_t tx) {
  GroupedWs w;
  // tiles of the narrowest class (which class a batch's full tiles are of depends on its T, P and E, and a
  // workspace serves every batch of no more slots), and a round of wide tiles split in two
  const uint32_t tt1 = (uint32_t)kClsCT[kNCls - 1] * (16 / tx), tt2 = (uint32_t)kClsCT[kNCls - 1] * (16 / 3);
  w.max_tiles1 = (uint32_t)(P / tt1 + E + 1) + kSplitRoom;
  w.max_tiles2 = (uint32_t)(P / tt2 + E + 1) + kSplitRoom;
  uint64_t o = 0;
  w.hdr = o; o += a256(sizeof(GroupedHdr));
  w.run = o; o += a256(4ull * ((uint64_t)T + 1));
  w.slot_tok = o; o += a256(4 * P);
  w.slot_w = o; o += a256(4 * P);
  w.ord = o; o += a256(4 * P);
  w.hist = o; o += a256(4ull * place_chunks(T, P) * E);
  w.sigma = o; o += a256(4 * P);  // per slot
  w.zeros = o; o += a256(hidden > inter ? hidden : inter);
  w.xq = o; o += a256((uint64_t)T * tx * hidden);
  w.aq = o; o += a256(P * 3 * inter);
  w.z = o; o += a256(P * 4 * hidden);
  // (these last: what comes before the B rows counts towards their 32-bit offsets, and so to the
  // largest batch accepted)
  w.tiles1 = o; o += a256(sizeof(Tile) * w.max_tiles1);
  w.tiles2 = o; o += a256(sizeof(Tile) * w.max_tiles2);
  w.tok_sigma = o; o += a256(4ull * T);
  w.total = o;
  return w;
}

// The two entries' shared body. Routes form (sel != null): plan, run and place build the slot list
// on the device from the routes. Slot-list form: the caller's expert ranges (start), tok, wt, ord
// and run; only the tiles are built here.
int grouped_body(const affx_layer* L, const void* x, const void* x_lo, uint32_t T, const uint32_t* sel,
                 const float* w, uint32_t K, const uint32_t* start, const uint32_t* tok, const float* wt,
                 const uint32_t* ord, const uint32_t* run, uint32_t n_slots, float* y, int accumulate,
                 void* ws, size_t ws_bytes, void* stream, const char* what) {
  if (!L || !x || !y || !ws || !L->base || !L->codebook) return set_error(AFFX_ERR_ARG, "%s: null pointer", what);
  if (L->n_experts == 0 || L->n_experts > AFFX_MAX_EXPERTS)
    return set_error(AFFX_DECLINED, "%s: n_experts must be 1..%d", what, AFFX_MAX_EXPERTS);
  if (L->hidden % kTileCols || L->inter % kTileCols || L->hidden == 0 || L->inter == 0 ||
      L->hidden > 8192 || L->inter > 8192)
    return set_error(AFFX_DECLINED, "%s: hidden and inter must be multiples of 1024, at most 8192", what);
  if (!(L->swiglu_limit > 0.f) || L->swiglu_limit > 1e6f)
    return set_error(AFFX_DECLINED, "%s: needs a SwiGLU clamp limit in (0, 1e6]", what);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(x_lo)) & 15u)
    return set_error(AFFX_ERR_ARG, "%s: x and x_lo must be 16-byte aligned", what);
  const uint32_t tx = x_lo ? 3 : 2;
  const uint64_t P = sel ? (uint64_t)T * K : n_slots;
  const GroupedWs lay = grouped_ws(T, P, L->n_experts, L->hidden, L->inter, tx);
  // the GEMM addresses its B rows with 32-bit offsets into the workspace
  if (P > (1ull << 31) || lay.aq + P * 3 * L->inter > (1ull << 32))
    return set_error(AFFX_DECLINED, "%s: batch too large (split it)", what);
  if (ws_bytes < lay.total)
    return set_error(AFFX_ERR_ARG, "%s: workspace %zu < %llu bytes", what, ws_bytes, (unsigned long long)lay.total);
  uint64_t off9[9];
  const uint64_t stride = affx_expert_layout(L->hidden, L->inter, off9, nullptr);
  if (L->stride < stride) return set_error(AFFX_ERR_ARG, "%s: layer stride below expert size", what);

  uint8_t* b = (uint8_t*)ws;
  hipStream_t s = (hipStream_t)stream;
  const uint32_t* slot_tok = sel ? (const uint32_t*)(b + lay.slot_tok) : tok;
  const float* slot_w = sel ? (const float*)(b + lay.slot_w) : wt;
  const uint32_t* ord_d = sel ? (const uint32_t*)(b + lay.ord) : ord;
  const uint32_t* run_d = sel ? (const uint32_t*)(b + lay.run) : run;
  GemmArgs A;
  A.base = (const uint8_t*)L->base;
  A.stride = L->stride;
  for (int i = 0; i < 9; ++i) A.off[i] = off9[i];
  A.hidden = L->hidden;
  A.inter = L->inter;
  A.codebook = (const uint32_t*)L->codebook;
  A.hdr = (const GroupedHdr*)(b + lay.hdr);
  A.slot_tok = slot_tok;
  A.n_sl = (uint32_t)P;
  A.n_tok = T;
  A.slot_sigma = (const int32_t*)(b + lay.sigma);
  A.ws = b;
  A.zero_off = lay.zeros;
  A.aq = b + lay.aq;
  A.z = (float*)(b + lay.z);
  A.limit = L->swiglu_limit;
  A.sigma_a = 7 - ilogbf(L->swiglu_limit * L->swiglu_limit);

  const uint32_t Pp = sel ? T * K : 0u;
  const uint32_t n_sl = (uint32_t)P;  // slot indices are below this (the routes form's taken slots too)
  const uint32_t zmax = L->hidden > L->inter ? L->hidden : L->inter;
  int32_t* tok_sigma = (int32_t*)(b + lay.tok_sigma);
  hipLaunchKernelGGL(grouped_prep_x_kernel, dim3(T), dim3(256), 0, s, (const uint16_t*)x, (const uint16_t*)x_lo,
                     L->hidden, tx, ord, run, n_sl, (int32_t*)(b + lay.sigma), tok_sigma, b + lay.xq,
                     (uint32_t*)(b + lay.zeros), zmax / 4);
  int rc = check_launch("grouped_prep_x_kernel");
  if (rc) return rc;
  // the GEMMs' grid: one workgroup per CU, a multiple of the 8 XCDs (the light class: two)
  int dev = 0, cus = 0;
  if ((rc = check_hip(hipGetDevice(&dev), "hipGetDevice"))) return rc;
  if ((rc = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute")))
    return rc;
  const uint32_t gmax = cus >= 8 ? (uint32_t)cus / 8u * 8u : 8u;
  const uint32_t k01 = widest_cls(T, P, L->n_experts, tx, L->inter / 128, gmax);
  const uint32_t k02 = widest_cls(T, P, L->n_experts, 3, L->hidden / 256, gmax);
  const PlanOut po{(GroupedHdr*)(b + lay.hdr), (Tile*)(b + lay.tiles1), (Tile*)(b + lay.tiles2),
                   lay.max_tiles1, lay.max_tiles2,
                   ClsGrid{L->inter / 128, gmax, 1.0f / (float)gmax,
                           light_cost(P, L->n_experts, k01, tx, L->inter / 128, gmax, L->hidden)},
                   ClsGrid{L->hidden / 256, gmax, 1.0f / (float)gmax,
                           light_cost(P, L->n_experts, k02, 3, L->hidden / 256, gmax, L->inter)}};
  uint32_t* hist = (uint32_t*)(b + lay.hist);
  if (sel && Pp <= kSmallPairs) {
    // one workgroup instead of three launches: 7.1 us against 5.4 + 8.2 + 5.0 at 144 pairs, 11.6 against
    // 5.2 + 8.4 + 5.4 at 1998, 13 to 15 from 3072 to 4096 against 4.8 + 8.1 + 6.2 at 5120 (kernel trace; the
    // gaps between launches come on top)
    hipLaunchKernelGGL(grouped_plan_small_kernel, dim3(1), dim3(kPlanThreads), 0, s, sel, w, Pp, T, K, L->n_experts,
                       k01, k02, tx, tok_sigma, (uint32_t*)(b + lay.slot_tok), (float*)(b + lay.slot_w),
                       (int32_t*)(b + lay.sigma), (uint32_t*)(b + lay.ord), (uint32_t*)(b + lay.run), po);
    if ((rc = check_launch("grouped_plan_small_kernel"))) return rc;
  } else {
    const uint32_t nch = sel ? (uint32_t)place_chunks(T, Pp) : 0u;
    if (sel) {
      hipLaunchKernelGGL(grouped_hist_kernel, dim3(nch), dim3(256), 0, s, sel, Pp, T, K, L->n_experts, hist,
                         (uint32_t*)(b + lay.run), (uint32_t*)(b + lay.ord));
      if ((rc = check_launch("grouped_hist_kernel"))) return rc;
    }
    hipLaunchKernelGGL(grouped_plan_kernel, dim3(1), dim3(kPlanThreads), 0, s, hist, nch, L->n_experts, k01, k02, tx,
                       sel ? nullptr : start, sel ? 0u : n_slots, po);
    if ((rc = check_launch("grouped_plan_kernel"))) return rc;
    if (sel) {
      hipLaunchKernelGGL(grouped_place_kernel, dim3(nch), dim3(256), 0, s, sel, w, Pp, K, L->n_experts,
                         (const uint32_t*)hist, tok_sigma, (uint32_t*)(b + lay.slot_tok), (float*)(b + lay.slot_w),
                         (int32_t*)(b + lay.sigma), (uint32_t*)(b + lay.ord));
      if ((rc = check_launch("grouped_place_kernel"))) return rc;
    }
  }
  // gate/up: 128 gate + 128 up rows per item; down: 256 rows. Items (row block, tile), the tile
  // count rounded up to a multiple of the 8 XCDs (see the kernel's order), run by a persistent
  // grid of one workgroup per CU (a multiple of 8), or fewer when there are fewer items
  // (the classes below the widest: at most one tile per expert, and the parts of split wide tiles)
  auto grid = [&](uint32_t row_blocks, uint32_t tiles, uint32_t per_cu) {
    const uint32_t items = row_blocks * ((tiles + 7) / 8 * 8);
    return items < per_cu * gmax ? items : per_cu * gmax;
  };
  A.tiles = (const Tile*)(b + lay.tiles1);
  A.max_tiles = lay.max_tiles1;
  A.b_off = lay.xq;
  auto each_cls = [&](auto ph, auto txc, uint32_t k0, const ClsGrid& cg, uint32_t max_tiles) {
    constexpr int PH = decltype(ph)::value, TX = decltype(txc)::value;
    const uint32_t part = L->n_experts + kSplitRoom < max_tiles ? L->n_experts + kSplitRoom : max_tiles;
    static_for<0, kNCls>([&](auto kc) {
      constexpr int k = decltype(kc)::value, CT = kClsCT[k];
      if ((uint32_t)k < k0 || (GTile<CT>::kLight && cg.light == 0u)) return;
      const dim3 g(grid(cg.nrb, (uint32_t)k == k0 ? max_tiles : part, GTile<CT>::kLight ? 2u : 1u));
      hipLaunchKernelGGL((grouped_gemm_kernel<PH, TX, CT>), g, dim3(kGT), 0, s, A);
    });
  };
  if (tx == 2)
    each_cls(IConst<0>{}, IConst<2>{}, k01, po.g1, lay.max_tiles1);
  else
    each_cls(IConst<0>{}, IConst<3>{}, k01, po.g1, lay.max_tiles1);
  if ((rc = check_launch("grouped_gemm_kernel (gate/up)"))) return rc;
  A.tiles = (const Tile*)(b + lay.tiles2);
  A.max_tiles = lay.max_tiles2;
  A.b_off = lay.aq;
  each_cls(IConst<1>{}, IConst<3>{}, k02, po.g2, lay.max_tiles2);
  if ((rc = check_launch("grouped_gemm_kernel (down)"))) return rc;
  hipLaunchKernelGGL(grouped_combine_kernel, dim3((L->hidden / 4 + 255) / 256, T), dim3(256), 0, s,
                     (const float*)(b + lay.z), ord_d, run_d, slot_w, n_sl, L->hidden, y, accumulate);
  return check_launch("grouped_combine_kernel");
}

}  // namespace

extern "C" {

size_t affx_grouped_workspace_size(uint32_t n_tok, uint32_t top_k, uint32_t n_experts,
                                   uint32_t hidden, uint32_t inter) {
  // sized for the 3-term gate/up input (x with a low part), the larger layout
  return (size_t)grouped_ws(n_tok, (uint64_t)n_tok * top_k, n_experts, hidden, inter, 3).total;
}

int affx_expert_ffn_grouped(const affx_layer* L, const void* x, const void* x_lo, uint32_t T,
                            const uint32_t* sel, const float* w, uint32_t K, float* y,
                            int accumulate, void* ws, size_t ws_bytes, void* stream) {
  if (!sel || !w) return set_error(AFFX_ERR_ARG, "ffn_grouped: null pointer");
  if (T == 0) return AFFX_OK;
  if (K == 0 || K > AFFX_MAX_TOPK)
    return set_error(AFFX_DECLINED, "ffn_grouped: top_k must be 1..%d", AFFX_MAX_TOPK);
  return grouped_body(L, x, x_lo, T, sel, w, K, nullptr, nullptr, nullptr, nullptr, nullptr, 0, y, accumulate, ws,
                      ws_bytes, stream, "ffn_grouped");
}

int affx_expert_ffn_grouped_slots(const affx_layer* L, const void* x, const void* x_lo, uint32_t T,
                                  const uint32_t* expert_start, const uint32_t* tok, const float* wt,
                                  const uint32_t* ord, const uint32_t* run, uint32_t n_slots, float* y,
                                  int accumulate, void* ws, size_t ws_bytes, void* stream) {
  if (!expert_start || !tok || !wt || !ord || !run) return set_error(AFFX_ERR_ARG, "ffn_grouped_slots: null pointer");
  if (T == 0) return AFFX_OK;
  return grouped_body(L, x, x_lo, T, nullptr, nullptr, 0, expert_start, tok, wt, ord, run, n_slots, y, accumulate,
                      ws, ws_bytes, stream, "ffn_grouped_slots");
}

}  // extern "C"
