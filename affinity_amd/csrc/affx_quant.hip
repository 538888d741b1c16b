// Producer side on the GPU: the synthetic-weight generator and the codebook quantiser.
//
// affx_quantize_matrix is the reference's quantize_matrix for the quad format
// (src/quant/blockquant.cpp:586-791) on the GPU, bit-exact: every float operation that decides an
// output is the reference's, in its order, with no contraction into FMAs. A block's setting (variant,
// scale, sign and rotation: up to 24, each the sum of four nearest-entry distances) is chosen in two
// stages. First every setting's error is taken from f32 matrix products with a bound on their
// rounding; where one setting's upper bound lies below all other lower bounds, that setting is the
// reference's choice, whatever the last bits. The rest (a few percent of the blocks: near ties, and
// inputs the bound does not cover) are settled by the reference's own search among the settings
// still open, exhaustively: each lane scores 16 of the 1024 entries, then a wave reduction keeps the
// minimum, which is exactly what the reference's scan and its acceleration grid return
// (src/quant/blockquant.cpp:162-174, 558-578). The codes of the chosen setting are the
// reference's scan, a quad a lane (the lowest index among equal minima).
//
// affx_gen_normal is the benchmark's synthetic generator: splitmix64 in counter form plus
// Box-Muller in double (the generator of src/quant/blockquant.cpp:37-42, 862-869), rounded to
// f32 and then to bf16.
#include "affx_common.h"

// Every float operation below is the reference's, one rounding each. HIP contracts a*b+c into an
// FMA by default, which moves distances by an ulp and flips near-tied nearest-code choices; the
// pragma turns that off for the code written in this file (the HIP headers' __fadd_rn family are
// plain operators compiled under the default, so they are not used here).
#pragma clang fp contract(off)

namespace affx {

// ---- generator ---------------------------------------------------------------------------------

__device__ __forceinline__ uint64_t splitmix_at(uint64_t seed, uint64_t k) {
  uint64_t x = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

__global__ void gen_normal_kernel(uint64_t seed, uint64_t n, double scale, float* __restrict__ out,
                                  int bf16_round) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double u1 = (double)((splitmix_at(seed, 2 * i) >> 11) + 1) * (1.0 / 9007199254740992.0);
  const double u2 = (double)((splitmix_at(seed, 2 * i + 1) >> 11) + 1) * (1.0 / 9007199254740992.0);
  const double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
  float f = (float)(scale * z);
  if (bf16_round) f = __uint_as_float((uint32_t)f32_to_bf16_rne(f) << 16);
  out[i] = f;
}

// ---- quantiser ---------------------------------------------------------------------------------

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
  return v;
}

// Squared distance of target t to entry e, dimensions summed in order, no contraction.
__device__ __forceinline__ float qdist(const float4 e, const float t0, const float t1,
                                       const float t2, const float t3) {
  const float a = e.x - t0, b = e.y - t1, c = e.z - t2, d = e.w - t3;
  float s = a * a;
  s = s + b * b;
  s = s + c * c;
  s = s + d * d;
  return s;
}

// Minimum distance of one quad target to the entries of one variant (wave-uniform result).
// The reference's scan starts from FLT_MAX and keeps strict improvements, so a minimum of
// FLT_MAX or more (or NaN) reads as FLT_MAX.
__device__ __forceinline__ float quad_min(const float4* __restrict__ ent, uint32_t lane, float t0,
                                          float t1, float t2, float t3) {
  float m = 3.402823466e38f;
#pragma unroll 4
  for (int j = 0; j < 16; ++j) {
    const float s = qdist(ent[lane + 64 * j], t0, t1, t2, t3);
    m = s < m ? s : m;
  }
  return wave_min(m);
}

// The scan's code of one quad: the lowest index among equal minima (wave-uniform result).
__device__ __forceinline__ uint32_t quad_argmin(const float4* __restrict__ ent, uint32_t lane, float t0, float t1,
                                                float t2, float t3) {
  float m = 3.402823466e38f;
  uint32_t bi = 0xFFFFFFFFu;
#pragma unroll 4
  for (int j = 0; j < 16; ++j) {
    const float s = qdist(ent[lane + 64 * j], t0, t1, t2, t3);
    if (s < m) { m = s; bi = lane + 64u * j; }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(m, o);
    const uint32_t oi = __shfl_xor(bi, o);
    if (ov < m || (ov == m && oi < bi)) { m = ov; bi = oi; }
  }
  return bi == 0xFFFFFFFFu ? 0u : bi;  // nothing below FLT_MAX: the scan's default, code 0
}

// The reference's setting search of one block (blockquant.cpp:706-762) among the settings of `open`
// (bit 12 v + 4 j + g: variant v, scale mid - 1 + j, g: bit 0 sign, bit 1 rotation), all lanes of
// the wave on one block: the first strict minimum in the order v, scale, g.
__device__ uint32_t search_block(const float4* ent, uint32_t lane, const float* __restrict__ blk,
                                 const float* __restrict__ imp, float rscale, int mid, uint32_t open) {
  float x[16], wt[4] = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = blk[i];
  if (imp) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float s = 0.f;
#pragma unroll
      for (int p = 0; p < 4; ++p) s = s + imp[4 * i + p];
      wt[i] = s / 4.0f;
    }
  }
  uint32_t best = 0;  // field: variant << 5 | g << 3 | scale
  double best_err = 1.7976931348623157e308;
  for (uint32_t v = 0; v < 2; ++v)
    for (int j = 0; j < 3; ++j) {
      const int s = mid - 1 + j;
      if (s < 0 || s > 7) continue;
      const float bs = rscale * (float)(1u << s);
      if (bs <= 0.f) continue;
      const float inv = 1.0f / bs;
      for (uint32_t g = 0; g < 4; ++g) {
        if (!((open >> (12u * v + 4u * j + g)) & 1u)) continue;
        const float sg = (g & 1u) ? -inv : inv;
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float t[4];
#pragma unroll
          for (int p = 0; p < 4; ++p) t[p] = ((g & 2u) ? x[4 * i + (p + 2) % 4] : x[4 * i + p]) * sg;
          const float d = quad_min(ent + v * kLut, lane, t[0], t[1], t[2], t[3]);
          acc = acc + d * wt[i];
        }
        const double e = (double)acc * (double)bs * (double)bs;
        if (e < best_err) { best_err = e; best = (v << 5) | (g << 3) | (uint32_t)s; }
      }
    }
  return best;
}

// ---- the search in matrix products -----------------------------------------------------------------
// Bound by VALU issue: the exhaustive search took 12 operations for every (entry, target) pair, 96
// targets a block; here a product and 8 minimum operations serve 512 of them, and the codes' scan
// is the only exhaustive one left. 2048 x 4096: 16.0 -> 3.05 ms (8.4M weights).
// A workgroup takes 1024 columns of a row, a wave 16 blocks of them. With t a quad's target, the
// distance to entry e is 2 (|e|^2 / 2 - e.t) + |t|^2: a 16x16x4 f32 product of 16 entries (A, row =
// entry) with the 16 blocks' targets (B, column = block, K = the quad's four dimensions) on top of
// C = |e|^2 / 2. The targets of the opposite sign are its negation, |e|^2 / 2 + e.t = |e|^2 - D, so 24
// products (3 scales x 2 rotations x 4 quads) an entry tile serve 48 of the 96 (setting, quad)
// pairs of a variant.
// Bound: u = 2^-24. The reference's float distance is within 6u of the true one; |e|^2 / 2 in f32,
// four products and four sums, each with one rounding of a value of at most |e|^2 / 2 + |e| |t| <=
// (E + |t|^2) (E = the largest |e|^2), are within 12u of that, twice it 24u; |t|^2 in f32 within 8u |t|^2;
// the sums over four quads with their weights (>= 0, else the block is searched in full) within
// 16u of themselves on either side. The code takes 44u (E + |t|^2) a quad and 64u of the sum.
// These are relative: a value below the normal range may be off by 2^-126 (2^-149 outside the matrix
// core) instead. With E > 1e-20 that is nothing beside 44u E, and a block whose weighted bound is not above
// 1e-30 (importances all but zero) is searched in full.
constexpr int kQuantMaxCols = 8192;
constexpr uint32_t kQuantChunk = 1024;
// A chunk of 64 columns (four blocks of a product's 16 columns, and one wave of the four) is searched in
// full, and so are rows of 128 where there are more of them than a device of 256 CUs holds workgroups of
// the products, three a CU. Both ways, us, products and full search: 64 columns, 512 rows 186 and 85, 2048
// rows 521 and 228; 128 columns, 512 rows 155 and 165, 768 rows 154 and 196, 1024 rows 300 and 243, 2048
// rows 521 and 448.
constexpr uint32_t kShort = 4;
constexpr uint32_t kAllRows = 3 * 256 + 1;
// Open settings of a wave's undecided blocks that it searches by itself: near ties leave two or three
// of a block's 24 open in a few percent of the blocks, a codebook of tied entries two in all 16.
constexpr uint32_t kOwnSettings = 64;
constexpr float kU = 5.9604645e-8f;
typedef float qv4f __attribute__((ext_vector_type(4)));

// Field i and code i of a chunk into their streams (zeroed; the bits are disjoint).
__device__ __forceinline__ void put_field(uint32_t* fbits, uint32_t i, uint32_t field) {
  const uint32_t at = i * 6;
  atomicOr(&fbits[at >> 5], field << (at & 31));
  if ((at & 31) > 26) atomicOr(&fbits[(at >> 5) + 1], field >> (32 - (at & 31)));
}
__device__ __forceinline__ void put_code(uint32_t* cbits, uint32_t i, uint32_t code) {
  const uint32_t at = i * 10;
  atomicOr(&cbits[at >> 5], code << (at & 31));
  if ((at & 31) > 22) atomicOr(&cbits[(at >> 5) + 1], code >> (32 - (at & 31)));
}
__device__ __forceinline__ float low_of(float a, float b) { return __builtin_fminf(a, b); }

// (kAll: every block is searched in full, which needs neither |e|^2 / 2 nor the products' registers, so a CU
// holds four workgroups and not three)
template <bool kAll>
__global__ void __launch_bounds__(256, kAll ? 4 : 3) quantize_rows_kernel(
    const float* __restrict__ w, uint32_t cols, uint32_t chunks, const float4* __restrict__ cb,
    const float* __restrict__ imp, uint8_t* __restrict__ codes, uint8_t* __restrict__ fields,
    uint16_t* __restrict__ rscales) {
  const uint32_t r = blockIdx.x / chunks, ch = blockIdx.x - r * chunks;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  __shared__ float4 ent[kVariants * kLut];                      // 32 KiB
  __shared__ __align__(16) float half[kAll ? 4 : kVariants * kLut];  // |e|^2 / 2
  __shared__ uint32_t cbits[kQuantChunk * 10 / 128];            // the chunk's code stream
  __shared__ uint32_t fbits[kQuantChunk * 6 / 512 + 1];         // the chunk's field stream
  __shared__ float red[8];
  __shared__ uint2 listed[kQuantChunk / kBlock];                // block | middle scale << 8, open settings
  __shared__ uint32_t n_listed;
  float e2max = 0.f;
  for (uint32_t i = tid; i < kVariants * kLut; i += 256) {
    const float4 e = cb[i];
    ent[i] = e;
    const float n = ((e.x * e.x + e.y * e.y) + e.z * e.z) + e.w * e.w;
    if constexpr (!kAll) half[i] = 0.5f * n;
    e2max = fmaxf(e2max, n < 1e30f ? n : INFINITY);  // (an entry past the bound, or a NaN, leaves no bound)
  }
  for (uint32_t i = tid; i < kQuantChunk * 10 / 128; i += 256) cbits[i] = 0;
  if (tid < kQuantChunk * 6 / 512 + 1) fbits[tid] = 0;
  if (tid == 0) n_listed = 0;

  const float* row = w + (uint64_t)r * cols;
  float rmax = 0.f;
  for (uint32_t c = tid; c < cols; c += 256) {
    const float a = fabsf(row[c]);
    rmax = rmax < a ? a : rmax;
  }
  rmax = -wave_min(-rmax);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    e2max = fmaxf(e2max, __shfl_xor(e2max, o));
  }
  if (lane == 0) { red[wv] = rmax; red[4 + wv] = e2max; }
  __syncthreads();
  rmax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
#pragma unroll
  for (int q = 0; q < 4; ++q) e2max = fmaxf(e2max, red[4 + q]);
  float rscale = rmax > 0.f ? ldexpf(rmax, -7) : 0.f;
  const uint16_t h = f32_to_bf16_rne(rscale);
  rscale = __uint_as_float((uint32_t)h << 16);
  if (ch == 0 && tid == 0) rscales[r] = h;

  // ---- this wave's 16 blocks: lane (c, kg) holds dimension kg of block c's quads ---------------------
  const uint32_t c0 = ch * kQuantChunk, nblk = min(cols - c0, kQuantChunk) / kBlock;
  const uint32_t c = lane & 15, kg = lane >> 4, b = 16u * wv + c;
  const bool live = b < nblk;
  const float* blk = row + c0 + (uint64_t)(live ? b : 0u) * kBlock;
  const float* bimp = imp ? imp + c0 + (live ? b : 0u) * kBlock : nullptr;
  float wq[4], wr[4], S[4], wt[4] = {1.f, 1.f, 1.f, 1.f}, bmax = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    wq[q] = live ? blk[4 * q + kg] : 0.f;
    wr[q] = __shfl_xor(wq[q], 32);  // dimension (kg + 2) % 4
    const float a = fabsf(wq[q]);
    bmax = bmax < a ? a : bmax;
    if (bimp) wt[q] = (((bimp[4 * q] + bimp[4 * q + 1]) + bimp[4 * q + 2]) + bimp[4 * q + 3]) * 0.25f;
  }
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    const float a = __shfl_xor(bmax, o);
    bmax = bmax < a ? a : bmax;
  }
  const bool need = live && bmax > 0.f && rscale > 0.f;
  int mid = 0;
  if (need) {
    const double ideal = (double)bmax / (double)rscale;
    double bd = 1.7976931348623157e308;
    for (int s = 0; s <= 7; ++s) {
      const double d = fabs((double)(float)(1u << s) - ideal);
      if (d < bd) { bd = d; mid = s; }
    }
  }
  float inv[3], er[3];
  uint32_t valid = 0;  // settings there are (scale 0..7), as in search_block
  const bool direct = kAll || nblk <= kShort;
  bool sane = !direct && e2max > 1e-20f && e2max < 1e30f;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int s = mid - 1 + j;
    const bool in = s >= 0 && s <= 7;
    const float bs = rscale * (float)(1u << (in ? s : 0));
    inv[j] = in && need ? 1.0f / bs : 0.f;
    if (in) valid |= 0xF00Fu << (4 * j);
    sane = sane && (!in || (bs > 1e-30f && bs < 1e30f));
  }
  // |t|^2 of the quads at the middle scale, of the scaled targets (the weights' own squares underflow);
  // four times that at the scale below, a quarter at the one above
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float t = wq[q] * inv[1];
    S[q] = t * t;
    S[q] = S[q] + __shfl_xor(S[q], 16);
    S[q] = S[q] + __shfl_xor(S[q], 32);
  }
  constexpr float kT2[3] = {4.f, 1.f, 0.25f};
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    er[j] = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) er[j] = er[j] + wt[q] * (44.f * kU * (e2max + S[q] * kT2[j]));
    er[j] = er[j] * (float)(1u << (2 * j));
    sane = sane && (!((valid >> (4 * j)) & 1u) || (er[j] > 1e-30f && er[j] < 1e30f));
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) sane = sane && wt[q] >= 0.f;

  uint32_t open = 0;
  if (!kAll && __ballot(need && sane)) {  // (the whole wave)
    float ea[24];  // errors of the settings over bs(j = 0)^2
    for (uint32_t v = 0; v < 2; ++v) {
      float m[24][2];
#pragma unroll
      for (int k = 0; k < 24; ++k) m[k][0] = m[k][1] = 3.402823466e38f;
      const float* A = reinterpret_cast<const float*>(ent + v * kLut) + 4u * c + kg;
      const float* Hf = half + v * kLut + 4u * kg;
#pragma unroll 1
      for (int i = 0; i < kLut / 16; ++i) {
        const float a = A[64 * i];
        const qv4f C = *reinterpret_cast<const qv4f*>(Hf + 16 * i);
        const qv4f n = C + C;
        auto product = [&](int k) -> qv4f {
          const float t = ((k / 4) % 2 ? wr[k % 4] : wq[k % 4]) * inv[k / 8];
          return __builtin_amdgcn_mfma_f32_16x16x4f32(a, -t, C, 0, 0, 0);
        };
        // (two products in flight: the minima of one run behind the next two)
        qv4f D0 = product(0), D1 = product(1);
#pragma unroll
        for (int k = 0; k < 24; ++k) {
          const qv4f D = D0;
          D0 = D1;
          if (k + 2 < 24) D1 = product(k + 2);
          __builtin_amdgcn_sched_barrier(0);
          m[k][0] = low_of(low_of(m[k][0], D[0]), D[1]);
          m[k][0] = low_of(low_of(m[k][0], D[2]), D[3]);
          m[k][1] = low_of(low_of(m[k][1], n[0] - D[0]), n[1] - D[1]);
          m[k][1] = low_of(low_of(m[k][1], n[2] - D[2]), n[3] - D[3]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int k = 0; k < 24; ++k)
#pragma unroll
        for (int sg = 0; sg < 2; ++sg) {
          float x = m[k][sg];
          x = low_of(x, __shfl_xor(x, 16));
          m[k][sg] = low_of(x, __shfl_xor(x, 32));
        }
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float e = 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            e = e + wt[q] * (2.f * m[8 * j + 4 * (g >> 1) + q][g & 1] + S[q] * kT2[j]);
          e = e * (float)(1u << (2 * j));
          if (v == 0) ea[4 * j + g] = e;
          else ea[12 + 4 * j + g] = e;
        }
    }
    float hi = 3.402823466e38f;
#pragma unroll
    for (int k = 0; k < 24; ++k)
      if ((valid >> k) & 1u) hi = low_of(hi, ea[k] + er[(k / 4) % 3] + 64.f * kU * fabsf(ea[k]));
#pragma unroll
    for (int k = 0; k < 24; ++k)
      if (((valid >> k) & 1u) && !(ea[k] - er[(k / 4) % 3] - 64.f * kU * fabsf(ea[k]) > hi)) open |= 1u << k;
  }
  if (!sane) open = valid;
  uint32_t field = 0;
  if (need && (open & (open - 1u)) == 0u && open != 0u) {
    const uint32_t k = (uint32_t)__builtin_ctz(open), j = (k % 12u) / 4u;
    field = ((k / 12u) << 5) | ((k & 3u) << 3) | (uint32_t)(mid - 1 + (int)j);
  }
  // the blocks left open, one at a time; where the chunk leaves a wave without blocks, a wave with many
  // settings open (not near ties, but blocks that the bound does not cover) lists its for the whole workgroup
  // instead, as a short chunk does all: in any order, a wave each in turn (512 x 512 with negative
  // importances, every block open: 1267 us with each wave at its own, 810 so; near ties listed too cost the
  // usual rows 2 %, as the waves then wait for each other twice)
  const bool undecided = need && (open & (open - 1u)) != 0u;
  uint64_t todo = __ballot(undecided && kg == 0u);
  bool shared = direct;
  if (todo && nblk <= 3u * kQuantChunk / kBlock / 4u) {
    uint32_t n = undecided && kg == 0u ? (uint32_t)__popc(open) : 0u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
    shared = shared || n > kOwnSettings;
  }
  const bool is_listed = live && shared && (direct || undecided);
  if (shared) {
    if (is_listed && kg == 0u) listed[atomicAdd(&n_listed, 1u)] = make_uint2(b | ((uint32_t)mid << 8), need ? open : 0u);
    todo = 0;
  }
  // (one loop over both: with a second call of the search in the kernel the search is slower by a third)
#pragma clang loop unroll(disable)
  for (int pass = 0;; ++pass) {
    for (uint32_t i = wv;; i += 4) {
      uint32_t bq, md, op;
      if (pass == 0) {
        if (!todo) break;
        const int src = __builtin_ctzll(todo);
        todo &= todo - 1;
        bq = 16u * wv + (uint32_t)src;
        md = (uint32_t)__shfl(mid, src);
        op = __shfl(open, src);
      } else {
        if (i >= n_listed) break;
        const uint2 q = listed[i];
        bq = __builtin_amdgcn_readfirstlane(q.x) & 255u;
        md = __builtin_amdgcn_readfirstlane(q.x) >> 8;
        op = __builtin_amdgcn_readfirstlane(q.y);
      }
      const uint32_t at = c0 + bq * kBlock;
      const uint32_t f = search_block(ent, lane, row + at, imp ? imp + at : nullptr, rscale, (int)md, op);
      if (pass == 0) {
        if (b == bq) field = f;
        continue;
      }
      if (lane == 0) put_field(fbits, bq, f);
      const float mag = rscale * (float)(1u << (f & 7u)), bs = (f & 8u) ? -mag : mag;
      if (!(mag > 0.f)) continue;
      const uint32_t rh = (f & 16u) ? 2u : 0u;
#pragma unroll
      for (uint32_t p = 0; p < 4; ++p) {
        const float* x = row + at + 4 * p;
        const uint32_t code = quad_argmin(ent + (f >> 5) * kLut, lane, x[rh] / bs, x[1 + rh] / bs, x[2 - rh] / bs, x[3 - rh] / bs);
        if (lane == 0) put_code(cbits, bq * 4 + p, code);
      }
    }
    if (pass == 0 && live && !is_listed) {
      // the codes: lane (c, kg) takes quad kg of block c
      const float mag = rscale * (float)(1u << (field & 7u));
      const float bs = (field & 8u) ? -mag : mag;
      const bool rot = (field & 16u) != 0u;
      uint32_t code = 0;
      if (mag > 0.f) {
        float x[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) x[p] = blk[4 * kg + p];
        const float t0 = (rot ? x[2] : x[0]) / bs, t1 = (rot ? x[3] : x[1]) / bs;
        const float t2 = (rot ? x[0] : x[2]) / bs, t3 = (rot ? x[1] : x[3]) / bs;
        const float4* ev = ent + (field >> 5) * kLut;
        float m = 3.402823466e38f;
#pragma unroll 8
        for (uint32_t e = 0; e < (uint32_t)kLut; ++e) {
          const float d = qdist(ev[e], t0, t1, t2, t3);
          if (d < m) { m = d; code = e; }
        }
      }
      if (kg == 0u) put_field(fbits, b, field);
      put_code(cbits, b * 4 + kg, code);
    }
    __syncthreads();
    if (pass == 1 || n_listed == 0) break;  // (the whole workgroup)
  }
  // 64 columns are whole bytes of both streams (20 and 3), and cols % 64 == 0
  const uint32_t ncb = nblk * 5, nfb = nblk * 3 / 4;
  const uint8_t* cs = reinterpret_cast<const uint8_t*>(cbits);
  const uint8_t* fs = reinterpret_cast<const uint8_t*>(fbits);
  uint8_t* co = codes + (uint64_t)r * (cols * 10 / 32) + ch * (kQuantChunk * 10 / 32);
  uint8_t* fo = fields + (uint64_t)r * (cols * 6 / 128) + ch * (kQuantChunk * 6 / 128);
  for (uint32_t i = tid; i < ncb; i += 256) co[i] = cs[i];
  for (uint32_t i = tid; i < nfb; i += 256) fo[i] = fs[i];
}

}  // namespace affx

using namespace affx;

extern "C" {

int affx_gen_normal(uint64_t seed, uint64_t n, double scale, void* out, int bf16_round,
                    void* stream) {
  if (!out) return set_error(AFFX_ERR_ARG, "gen_normal: null output");
  if (n == 0) return AFFX_OK;
  const uint64_t blocks = (n + 255) / 256;
  if (blocks > 0x7FFFFFFFull) return set_error(AFFX_ERR_ARG, "gen_normal: n too large");
  hipLaunchKernelGGL(gen_normal_kernel, dim3((uint32_t)blocks), dim3(256), 0, (hipStream_t)stream,
                     seed, n, scale, (float*)out, bf16_round);
  return check_launch("gen_normal_kernel");
}

int affx_quantize_matrix(const void* w, uint32_t rows, uint32_t cols, const void* codebook_f32,
                         const void* importance, void* codes, void* fields, void* rscales,
                         void* stream) {
  if (!w || !codebook_f32 || !codes || !fields || !rscales)
    return set_error(AFFX_ERR_ARG, "quantize_matrix: null pointer");
  if (rows == 0 || cols == 0 || cols % 64 || cols > kQuantMaxCols)
    return set_error(AFFX_ERR_ARG, "quantize_matrix: cols must be a multiple of 64 and <= %d",
                     kQuantMaxCols);
  const uint32_t chunks = (cols + kQuantChunk - 1) / kQuantChunk;
  const bool all = cols <= 64 || (cols <= 128 && rows >= kAllRows);
  auto* kernel = all ? quantize_rows_kernel<true> : quantize_rows_kernel<false>;
  // (a launch holds at most 2^32 threads: a matrix of millions of long rows takes several)
  const uint32_t slab = (1u << 23) / chunks;
  for (uint32_t r0 = 0; r0 < rows;) {
    const uint32_t n = rows - r0 < slab ? rows - r0 : slab;
    hipLaunchKernelGGL(kernel, dim3(n * chunks), dim3(256), 0, (hipStream_t)stream,
                       (const float*)w + (uint64_t)r0 * cols, cols, chunks, (const float4*)codebook_f32,
                       (const float*)importance, (uint8_t*)codes + (uint64_t)r0 * (cols / 32u * 10u),
                       (uint8_t*)fields + (uint64_t)r0 * (cols / 64u * 3u), (uint16_t*)rscales + r0);
    if (int rc = check_launch("quantize_rows_kernel")) return rc;
    r0 += n;
  }
  return AFFX_OK;
}

// One synthetic expert in container layout: gate/up/down = bf16(0.02 * N(0,1)) with seeds
// seed + 0/1/2, quantised against `codebook_f32`. `scratch` holds rows*cols floats of the largest
// matrix (inter*hidden).
int affx_fill_expert(void* expert, uint64_t hidden, uint64_t inter, const void* codebook_f32,
                     uint32_t seed, void* scratch, void* stream) {
  if (!expert || !codebook_f32 || !scratch) return set_error(AFFX_ERR_ARG, "fill_expert: null pointer");
  uint64_t off[9];
  affx_expert_layout(hidden, inter, off, nullptr);
  const uint64_t rows[3] = {inter, inter, hidden}, cols[3] = {hidden, hidden, inter};
  uint8_t* e = (uint8_t*)expert;
  for (int m = 0; m < 3; ++m) {
    int rc = affx_gen_normal((uint64_t)seed + m, rows[m] * cols[m], 0.02, scratch, 1, stream);
    if (rc) return rc;
    rc = affx_quantize_matrix(scratch, (uint32_t)rows[m], (uint32_t)cols[m], codebook_f32, nullptr,
                              e + off[3 * m], e + off[3 * m + 1], e + off[3 * m + 2], stream);
    if (rc) return rc;
  }
  return AFFX_OK;
}

}  // extern "C"
