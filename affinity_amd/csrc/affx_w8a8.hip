// The reference's single-matrix W8A8 GEMM over tiles of routed tokens, for a caller that drives
// its batch pipeline step by step (expert_gemm_wmma_hip, src/gpu/expert_kernel_hip.h:217-228;
// kernel src/gpu/expert_kernel.hip:364-825, host 3018-3062). For every tile (one expert matrix,
// nt <= 64 tokens of the chunk) and every row r:
//   y[r][j] = bf16(rs[r]) * wscale * out,  out = fma-fold over the 128-column blocks kb, in order,
//             of raw_kb * xs[t][kb],  raw_kb = sum over the block of W8[r][k] * x8[t][k]
// (expert_kernel.hip:808-818 for the fold, 820-837 for the row scale), t = tok ? tok[j] : j. W8 is
// the weight's E4M3 value without its row scale, x8 the E4M3 activation, xs its f32 scale per
// (token, 128-column block).
//
// A wave decodes the column tiles of a 16-row wave tile into MFMA A fragments (the decode's LDS
// codebook and step order). In a fragment of the wave tile lane group g holds 32 columns of segment g,
// so one MFMA's 128 values of K would span four 128-column blocks, whose sums must stay apart. Four
// steps' fragments are a 4 x 4 matrix of (segment, 32 columns) over (lane group, fragment): transposed
// by lane-row swaps (32 VALU operations for 4 fragments), lane group j of fragment g holds
// columns 32 j .. of segment g's block, and an MFMA is one block of 16 tokens. Its sums are
// folded into the outputs in block order, one fma each. (Without the transposition each MFMA took a
// quad of tokens, its B zero outside the group: four times the MFMAs, and a fold through DPP quad
// broadcasts: 256 tokens' steps over 256 experts 1092 us, now 672.)
//
// An item is 128 rows (64 where the launch has few) by at most 16 tokens (one MFMA column tile) of a
// tile, a wave for 16 rows: most tiles of
// a batch of a few hundred tokens over 256 experts have no more, and the weights' stream and the
// decode are the bound, so a persistent workgroup requests its next column tile's or next item's
// weights and token rows before it decodes the current ones, two workgroups (16 waves) a CU. A tile
// of more tokens is several items, which decode the same weights again. (A second kernel for the tiles
// of more than 16 tokens, one decode held for all their products at half the waves a CU, made the
// 256-token steps 755 us against 672: a handful of such tiles fills a launch of its own badly.)
// Full tiles: 384 of 64 tokens, 2048 x 4096, 1.69 -> 1.23 ms (334 TFLOP/s); 256 of one token 987 -> 191 us.
#include "affx_lut.h"

namespace affx {

constexpr int kW8Waves = 8;           // waves of a workgroup (half of them in launches of few items)
constexpr int kW8KC = 2;              // codebook copies
constexpr uint32_t kW8MaxTok = 64;    // the reference's kExpertWmmaTok (expert_kernel_hip.h:195)
constexpr uint32_t kW8Row = kTileCols + 16u;  // LDS bytes of one staged token row (padded)

struct W8a8Args {
  const affx_expert_tile* tiles;
  const uint8_t* x8;
  const float* xs;
  const uint32_t* codebook;
  uint32_t rows, cols, cap, items;  // (items: tiles x row blocks x token groups of the cap)
  float wscale;
  int y_bf16;
};

__device__ __forceinline__ uint16_t w8_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// A tile's tokens: at most `cap` (the launch's max_nt rounded up to a power of two of quads; a tile
// past the launch's max_nt is out of contract and cut there). The launch list is not written while
// a kernel runs: scalar loads.
__device__ __forceinline__ uint32_t w8_tokens(const affx_expert_tile* tiles, uint32_t tile, uint32_t cap) {
  return min(*AFFX_CONST_PTR(uint32_t, &tiles[tile].nt), cap);
}
// Token row of tile column j.
__device__ __forceinline__ uint32_t w8_row(const uint32_t* tok, uint32_t j) {
  return tok ? *AFFX_CONST_PTR(uint32_t, tok + j) : j;
}

// Transposes four steps' fragments of a half (steps 4h .. 4h + 3): f[j] of lane group g, the half's
// columns 32 j .. of segment g, becomes f[g] of lane group j.
__device__ __forceinline__ void w8_transpose(v8i (&f)[4]) {
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const auto p = __builtin_amdgcn_permlane32_swap((uint32_t)f[0][d], (uint32_t)f[2][d], false, false);
    const auto q = __builtin_amdgcn_permlane32_swap((uint32_t)f[1][d], (uint32_t)f[3][d], false, false);
    const auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const auto t = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    f[0][d] = (int)r[0];
    f[1][d] = (int)r[1];
    f[2][d] = (int)t[0];
    f[3][d] = (int)t[1];
  }
}
// The four fragments of half h of the unit, one block of 128 columns each.
__device__ __forceinline__ void w8_half(Unit& u, const uint8_t* lut, uint32_t copy4, int h, v8i (&f)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t raw[8], bv[2];
    pin_step(u, 4 * h + j);
    lut_lookup_step<kW8KC, true>(u, lut, nullptr, copy4, 4 * h + j, raw, bv);
    f[j] = lut_finish(raw, bv);
    asm volatile("" ::: "memory");  // (one step's table reads in flight at a time: registers)
  }
  w8_transpose(f);
}
// B of block kb (of the column tile's eight) for the lane's token, whose staged row this is.
__device__ __forceinline__ v8i w8_b(const uint8_t* row, uint32_t kg, int kb) {
  return b_step(reinterpret_cast<const u32x4*>(row + kg * 32u + 128u * kb), 0);
}
// Folds the eight blocks' sums of a column tile, res[h][g] of block 2 g + h, in block order; sc: the
// lane's token's scales of the eight blocks.
__device__ __forceinline__ void w8_fold(const v4f (&res)[2][4], const float* sc, float (&out)[4]) {
  const float4 s0 = *reinterpret_cast<const float4*>(sc);
  const float4 s1 = *reinterpret_cast<const float4*>(sc + 4);
  const float s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
  for (int kb = 0; kb < 8; ++kb)
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = __builtin_fmaf(res[kb & 1][kb >> 1][v], s[kb], out[v]);
}

// Writes the lane's results of token column j: y[row][j] for its four rows.
__device__ __forceinline__ void w8_store(const W8a8Args& A, void* y, uint32_t ld, uint32_t row0, uint32_t j,
                                         const float (&out)[4], uint2 rsv) {
  const float rs[4] = {__uint_as_float(rsv.x << 16) * A.wscale, __uint_as_float(rsv.x & 0xFFFF0000u) * A.wscale,
                       __uint_as_float(rsv.y << 16) * A.wscale, __uint_as_float(rsv.y & 0xFFFF0000u) * A.wscale};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const uint64_t at = (uint64_t)(row0 + v) * ld + j;
    const float val = out[v] * rs[v];
    if (A.y_bf16)
      reinterpret_cast<uint16_t*>(y)[at] = w8_bf16(val);
    else
      reinterpret_cast<float*>(y)[at] = val;
  }
}

// An item: NW row tiles (one a wave) of a tile's tokens j0 .. j0 + n - 1.
struct W8Item {
  const uint8_t* codes;
  const uint8_t* fields;
  const uint32_t* tok;
  uint32_t tile, j0, n, rt;
};
// Item order: tile, row block, token group (nch groups of kW8Cols tokens; adjacent items, which run at
// the same time, read the same weights). Most tiles fill the first group only, so workgroup b takes
// item r G + (b + r) % G in round r (G the grid): its items go through the groups in turn, not
// through one (G is a multiple of nch).
constexpr uint32_t kW8Cols = 16;
struct W8Order {
  uint32_t nrb, nch, items;
};
// (the lane is counted where it is used: lane values held across the steps were spilled, and a
// reload, a vector memory load, waits for every load in flight)
__device__ __forceinline__ uint32_t w8_lane() {
  uint32_t z = 0u;
  AFFX_PIN(z);
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
}
// The first item in use from round r on (advanced); false past the last. Four rounds (a tile's token groups) are looked at by
// scalar loads, from there 64 at a time, a lane each: a list of mostly pads has hundreds of rounds without
// an item (4096 pads, 2048 rows: 282 us by scalar loads alone, now 7.4).
template <int NW>
__device__ __forceinline__ bool w8_seek(const W8a8Args& A, const W8Order& o, uint32_t& r, uint32_t wv, W8Item& I) {
  for (uint32_t tries = 0; (uint64_t)r * gridDim.x < o.items; ++tries) {
    if (tries >= 4u) {
      const uint32_t rl = r + w8_lane(), il = rl * gridDim.x + (blockIdx.x + rl) % gridDim.x;
      bool used = il < o.items;
      if (used) {
        const uint32_t ql = il / o.nch;
        used = (il - ql * o.nch) * kW8Cols < min(A.tiles[ql / o.nrb].nt, A.cap);
      }
      const uint64_t m = __ballot(used);
      if (m == 0u) {
        r += 64u;
        continue;
      }
      r += (uint32_t)__builtin_ctzll(m);
    }
    r = __builtin_amdgcn_readfirstlane(r);
    const uint32_t it = r * gridDim.x + (blockIdx.x + r) % gridDim.x;
    const uint32_t q = it / o.nch, j0 = (it - q * o.nch) * kW8Cols, tile = q / o.nrb;
    const uint32_t nt = it < o.items ? w8_tokens(A.tiles, tile, A.cap) : 0u;
    if (j0 >= nt) {
      ++r;
      continue;
    }
    I.tile = __builtin_amdgcn_readfirstlane(tile);
    I.j0 = __builtin_amdgcn_readfirstlane(j0);
    const affx_expert_tile* T = A.tiles + I.tile;
    I.codes = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->codes));
    I.fields = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->fields));
    I.tok = reinterpret_cast<const uint32_t*>(*AFFX_CONST_PTR(uint64_t, &T->tok));
    I.n = __builtin_amdgcn_readfirstlane(min(nt - j0, kW8Cols));
    I.rt = __builtin_amdgcn_readfirstlane((q - tile * o.nrb) * NW + wv);
    return true;
  }
  return false;
}
// The lane's four accumulator rows' scales.
__device__ __forceinline__ uint2 w8_rscales(const W8a8Args& A, const W8Item& I, uint32_t kg) {
  return *reinterpret_cast<const uint2*>(
      reinterpret_cast<const uint16_t*>(*AFFX_CONST_PTR(uint64_t, &A.tiles[I.tile].rscales)) + I.rt * 16u + 4u * kg);
}
__device__ __forceinline__ void* w8_y(const W8a8Args& A, const W8Item& I, uint32_t& ld) {
  const affx_expert_tile* T = A.tiles + I.tile;
  const uint32_t l = *AFFX_CONST_PTR(uint32_t, &T->ld);
  ld = l ? l : *AFFX_CONST_PTR(uint32_t, &T->nt);
  return reinterpret_cast<void*>(*AFFX_CONST_PTR(uint64_t, &T->y));
}
// Stages one token of a column tile: its 1 KiB of activations (one direct-to-LDS instruction) and its
// eight scales.
__device__ __forceinline__ void w8_stage(const W8a8Args& A, const W8Item& I, uint32_t ct, uint32_t j, uint32_t lane,
                                         uint8_t* row, float* sc) {
  const uint32_t t = w8_row(I.tok, j);
  const __amdgpu_buffer_rsrc_t r = buffer_rsrc(A.x8 + (uint64_t)t * A.cols + (uint64_t)ct * kTileCols, kTileCols);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, AFFX_LDS_PTR(row), 16, lane * 16u, 0, 0, 0);
  const __amdgpu_buffer_rsrc_t q = buffer_rsrc(A.xs + (uint64_t)t * (A.cols / 128u) + ct * 8u, 32u);
  if (lane < 8u) __builtin_amdgcn_raw_ptr_buffer_load_lds(q, AFFX_LDS_PTR(sc), 4, lane * 4u, 0, 0, 0);
}
// LDS: the codebook and two buffers of a column tile's token rows and scales, so two workgroups a CU (at
// most 128 registers a wave). The steps of a workgroup are (item, column tile) pairs in order; each
// step first requests the next step's unit and token rows, then decodes and multiplies its own, and
// ends in one barrier.
template <int NW>
__global__ void __launch_bounds__(NW * 64, NW / 2) w8a8_gemm_kernel(W8a8Args A) {
  constexpr int kW8T = NW * 64;
  __shared__ __align__(16) uint32_t lut_s[Lut<kW8KC, true>::kDwords];
  // (two arrays a kind: the compiler can tell the buffer being read from the one being written)
  __shared__ __align__(16) uint8_t xb0[kW8Cols * kW8Row], xb1[kW8Cols * kW8Row];
  __shared__ __align__(16) float xs0[kW8Cols * 8], xs1[kW8Cols * 8];
  const uint8_t* lut = reinterpret_cast<const uint8_t*>(lut_s);
  const uint32_t tid = threadIdx.x;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nct = A.cols / kTileCols, nrt = A.rows / kTileRows;
  const W8Order o{(nrt + NW - 1) / NW, A.cap > kW8Cols ? A.cap / kW8Cols : 1u, A.items};
  // The codebook: in a launch of few items first, as it waits for no descriptor (one tile of one token, 2048 x
  // 1024, 5.1 us with it after the weights, 4.7 so; 2048 x 4096 11.0 and 10.7), else after the first weights,
  // which are the bound (64 tiles of 5 tokens, 4096 x 2048, 49.1 us and 51.2 with it first).
  constexpr int kPer = 2048 / kW8T;
  uint32_t cbv[kPer];
  auto codebook = [&]() {
#pragma unroll
    for (int i = 0; i < kPer; ++i) cbv[i] = A.codebook[tid + (uint32_t)i * kW8T];
  };
  if constexpr (NW < kW8Waves) codebook();
  uint32_t r = 0;
  W8Item I;
  if (!w8_seek<NW>(A, o, r, wv, I)) return;  // (the whole workgroup)
  auto stage = [&](const W8Item& J, uint32_t ct, uint8_t* xb, float* xs) {
#pragma unroll
    for (uint32_t j = wv; j < kW8Cols; j += NW)
      if (j < J.n) w8_stage(A, J, ct, J.j0 + j, w8_lane(), xb + j * kW8Row, xs + j * 8u);
  };
  auto load = [&](Unit& u, const W8Item& J, uint32_t ct) {
    if (J.rt < nrt) load_unit_ordered(u, J.codes, J.fields, (uint64_t)J.rt * nct + ct, w8_lane());
  };

  Unit ua, ub;
  load(ua, I, 0);
  stage(I, 0, xb0, xs0);
  if constexpr (NW == kW8Waves) codebook();
  build_lut<kW8KC, kW8T, kPer, true>(lut_s, cbv, tid);
  __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
  __syncthreads();

  float out[4] = {};
  uint32_t ct = 0;
  // one step, of unit u from buffers (xb, xs), with the next step's going to un and (yb, ys); false
  // after the last
  auto step = [&](Unit& u, Unit& un, const uint8_t* xb, const float* xs, uint8_t* yb, float* ys) -> bool {
    const bool last = ct + 1 == nct;
    W8Item N = I;
    bool more = true;
    if (last) more = w8_seek<NW>(A, o, ++r, wv, N);
    const bool rows_ok = I.rt < nrt;
    const uint32_t lane = w8_lane(), c = lane & 15, kg = lane >> 4, copy4 = ((lane >> 1) & (kW8KC - 1)) * 4u;
    // (requested here, used after the last column tile's products)
    uint2 rsv = {0u, 0u};
    if (last && rows_ok) rsv = w8_rscales(A, I, kg);
    if (more) {
      load(un, N, last ? 0u : ct + 1u);
      stage(N, last ? 0u : ct + 1u, yb, ys);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (rows_ok) {
      // (a column past the item's tokens multiplies what its row of the LDS holds and is not stored)
      v4f res[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v8i f[4];
        w8_half(u, lut, copy4, h, f);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          res[h][g] = mfma(f[g], w8_b(xb + c * kW8Row, kg, 2 * g + h), v4f{0.f, 0.f, 0.f, 0.f});
          asm volatile("" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      w8_fold(res, xs + c * 8u, out);
    }
    if (last) {
      if (rows_ok && c < I.n) {
        uint32_t ld;
        void* y = w8_y(A, I, ld);
        w8_store(A, y, ld, I.rt * 16u + 4u * kg, I.j0 + c, out, rsv);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) out[v] = 0.f;
    }
    if (!more) return false;
    I = N;
    ct = last ? 0u : ct + 1u;
    __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
    __syncthreads();
    return true;
  };
  while (step(ua, ub, xb0, xs0, xb1, xs1) && step(ub, ua, xb1, xs1, xb0, xs0)) {
  }
}

}  // namespace affx

using namespace affx;

extern "C" int affx_expert_gemm_w8a8(const affx_expert_tile* tiles, uint32_t n_tiles, uint32_t max_nt, const void* x8,
                                     const float* xs, const uint32_t* codebook, uint32_t rows, uint32_t cols,
                                     float wscale, int y_bf16, void* stream) {
  if (n_tiles == 0) return AFFX_OK;
  if (!tiles || !x8 || !xs || !codebook) return set_error(AFFX_ERR_ARG, "expert_gemm_w8a8: null pointer");
  if (rows == 0 || rows % kTileRows || cols == 0 || cols % kTileCols || max_nt == 0 || max_nt > kW8MaxTok ||
      n_tiles > 65535u || (uint64_t)rows * cols > 0xFFFFFFFFull)
    return set_error(AFFX_DECLINED, "expert_gemm_w8a8: needs rows %% 16 == 0, cols a multiple of 1024, 1 <= max_nt "
                     "<= %u and at most 65535 tiles (got %u x %u, max_nt %u, %u tiles)", kW8MaxTok, rows, cols,
                     max_nt, n_tiles);
  if ((reinterpret_cast<uintptr_t>(x8) | reinterpret_cast<uintptr_t>(xs)) & 15u)
    return set_error(AFFX_ERR_ARG, "expert_gemm_w8a8: x8 and xs must be 16-byte aligned");
  W8a8Args A;
  A.tiles = tiles;
  A.x8 = (const uint8_t*)x8;
  A.xs = xs;
  A.codebook = codebook;
  A.rows = rows;
  A.cols = cols;
  A.wscale = wscale;
  A.y_bf16 = y_bf16 ? 1 : 0;
  const uint32_t nq = (max_nt + 3u) / 4u;
  A.cap = nq <= 1 ? 4u : nq <= 2 ? 8u : nq <= 4 ? 16u : nq <= 8 ? 32u : 64u;
  const uint32_t nch = A.cap > kW8Cols ? A.cap / kW8Cols : 1u;
  const uint64_t items = (uint64_t)n_tiles * ((rows / kTileRows + kW8Waves - 1) / kW8Waves) * nch;
  if (items > 0x7FFFFFFFull) {
    // (a matrix of over a million rows: half the tiles at a time)
    int rc = affx_expert_gemm_w8a8(tiles, n_tiles / 2, max_nt, x8, xs, codebook, rows, cols, wscale, y_bf16, stream);
    return rc ? rc : affx_expert_gemm_w8a8(tiles + n_tiles / 2, n_tiles - n_tiles / 2, max_nt, x8, xs, codebook, rows,
                                           cols, wscale, y_bf16, stream);
  }
  int dev = 0, cus = 0, rc;
  if ((rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) ||
      (rc = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute")))
    return rc;
  // A launch of few items is bound by one item's latency: where there is a CU for each half of them, items
  // of 64 rows (a wave a SIMD: one token, 2048 x 4096, 14.1 us in items of 128 rows, 10.7 so).
  const uint64_t half = (uint64_t)n_tiles * ((rows / kTileRows + kW8Waves / 2 - 1) / (kW8Waves / 2)) * nch;
  const bool few = half <= (uint64_t)(cus > 0 ? cus : 1) && half > items;
  A.items = (uint32_t)(few ? half : items);
  // persistent: as many workgroups as the device holds at once, a multiple of the token groups
  const uint32_t most = 2u * (uint32_t)(cus > 1 ? cus / 2 * 2 : 2);
  const uint32_t grid = A.items < most ? A.items : most;
  if (few)
    hipLaunchKernelGGL((w8a8_gemm_kernel<kW8Waves / 2>), dim3(grid), dim3(kW8Waves * 32), 0, (hipStream_t)stream, A);
  else
    hipLaunchKernelGGL((w8a8_gemm_kernel<kW8Waves>), dim3(grid), dim3(kW8Waves * 64), 0, (hipStream_t)stream, A);
  return check_launch("w8a8_gemm_kernel");
}
