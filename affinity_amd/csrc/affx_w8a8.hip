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
// codebook and step order). One MFMA step's 128 K values span four 128-column blocks (lane group g
// holds 32 columns of the tile's segment g), so to keep the blocks' sums apart the B operand places
// the columns of group g of a token in B column 4 (token of the quad) + g and zeros elsewhere: one
// MFMA gives, for four tokens, each group's partial, steps 0-3 completing block 2g of the tile and
// steps 4-7 block 2g + 1. A (row, token)'s eight partials then sit in one lane quad, and every lane
// of the quad folds them in block order (DPP quad broadcasts).
//
// Tiles run in two persistent kernels by their token count, which only the device knows: each
// kernel's workgroups walk the whole list and pass over the other's tiles (a scalar load each).
//  * light tiles (at most 8 tokens; most tiles of a batch of a few hundred tokens over 256
//    experts): bound by the weights' stream, so 16 waves a CU keep two units a wave in flight, and
//    a workgroup's next column tile or next item is requested before the current one is decoded;
//  * heavy tiles: bound by the MFMAs (each issued for one column group of a token quad), so a
//    tile's decode is kept for all its quads, as many as its tokens fill.
#include "affx_lut.h"

namespace affx {

constexpr int kW8Waves = 4;
constexpr int kW8T = kW8Waves * 64;
constexpr int kW8KC = 2;              // codebook copies
constexpr uint32_t kW8MaxTok = 64;    // the reference's kExpertWmmaTok (expert_kernel_hip.h:195)
constexpr uint32_t kW8Row = kTileCols + 16u;  // LDS bytes of one staged token row (padded)

struct W8a8Args {
  const affx_expert_tile* tiles;
  const uint8_t* x8;
  const float* xs;
  const uint32_t* codebook;
  uint32_t rows, cols, n_tiles, cap;
  float wscale;
  int y_bf16;
};

__device__ __forceinline__ uint16_t w8_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// value of lane G of this lane's quad (DPP quad_perm [G, G, G, G])
template <int G>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), G * 0x55, 0xF, 0xF, false));
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

// Folds one quad's partials of a column tile into out, block 2g + h of the tile: group g's partial
// (lane g of the quad, a DPP quad broadcast), half h; sc: the token's scales of the eight blocks.
__device__ __forceinline__ void w8_fold(const v4f& acc0, const v4f& acc1, const float* sc, float (&out)[4]) {
  const float4 s0 = *reinterpret_cast<const float4*>(sc);
  const float4 s1 = *reinterpret_cast<const float4*>(sc + 4);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float o = out[v];
    o = __builtin_fmaf(quad_lane<0>(acc0[v]), s0.x, o);
    o = __builtin_fmaf(quad_lane<0>(acc1[v]), s0.y, o);
    o = __builtin_fmaf(quad_lane<1>(acc0[v]), s0.z, o);
    o = __builtin_fmaf(quad_lane<1>(acc1[v]), s0.w, o);
    o = __builtin_fmaf(quad_lane<2>(acc0[v]), s1.x, o);
    o = __builtin_fmaf(quad_lane<2>(acc1[v]), s1.y, o);
    o = __builtin_fmaf(quad_lane<3>(acc0[v]), s1.z, o);
    o = __builtin_fmaf(quad_lane<3>(acc1[v]), s1.w, o);
    out[v] = o;
  }
}

// Writes one quad's results (the lanes of c % 4 == 0): y[row][j] for the lane's four rows.
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

// ---- light tiles: at most kW8Light tokens -------------------------------------------------------
// Eight waves, 128 rows of a tile an item; LDS: the codebook and two buffers of a column tile's
// token rows and scales, so two workgroups a CU (at most 128 registers a wave). The steps of a
// workgroup are (item, column tile) pairs in order; each step first requests the next step's unit
// and token rows, then decodes and multiplies its own, and ends in one barrier.
constexpr uint32_t kW8Light = 8;
constexpr int kW8LWaves = 8;
constexpr int kW8LT = kW8LWaves * 64;
static_assert(kW8Light == (uint32_t)kW8LWaves, "wave w stages token row w");

__global__ void __launch_bounds__(kW8LT, 4) w8a8_light_kernel(W8a8Args A) {
  __shared__ __align__(16) uint32_t lut_s[Lut<kW8KC, true>::kDwords];
  // (two arrays a kind: the compiler can tell the buffer being read from the one being written)
  __shared__ __align__(16) uint8_t xb0[kW8Light * kW8Row], xb1[kW8Light * kW8Row];
  __shared__ __align__(16) float xs0[kW8Light * 8], xs1[kW8Light * 8];
  __shared__ __align__(16) uint8_t zero_s[kSegCols];  // B of the lanes outside a token's column group
  const uint8_t* lut = reinterpret_cast<const uint8_t*>(lut_s);
  const uint32_t tid = threadIdx.x;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (the lane is counted where it is used: lane values held across the steps were spilled, and a
  // reload, a vector memory load, waits for every load in flight)
  auto lane_now = [&]() -> uint32_t {
    uint32_t z = 0u;
    AFFX_PIN(z);
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
  };
  const uint32_t nct = A.cols / kTileCols, nkb = A.cols / 128u, nrt = A.rows / kTileRows;
  const uint32_t nrb = (nrt + kW8LWaves - 1) / kW8LWaves, items = A.n_tiles * nrb;
  auto seek = [&](uint32_t it) -> uint32_t {
    for (; it < items; it += gridDim.x) {
      const uint32_t nt = w8_tokens(A.tiles, it / nrb, A.cap);
      if (nt != 0 && nt <= kW8Light) break;
    }
    return __builtin_amdgcn_readfirstlane(it);
  };
  struct Item {
    const uint8_t* codes;
    const uint8_t* fields;
    const uint32_t* tok;
    uint32_t tile, n, rt;
  };
  auto open = [&](uint32_t it) -> Item {
    Item I;
    I.tile = __builtin_amdgcn_readfirstlane(it / nrb);
    const affx_expert_tile* T = A.tiles + I.tile;
    I.codes = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->codes));
    I.fields = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->fields));
    I.tok = reinterpret_cast<const uint32_t*>(*AFFX_CONST_PTR(uint64_t, &T->tok));
    I.n = __builtin_amdgcn_readfirstlane(w8_tokens(A.tiles, I.tile, A.cap));
    I.rt = __builtin_amdgcn_readfirstlane((it - I.tile * nrb) * kW8LWaves + wv);
    return I;
  };
  uint32_t it = seek(blockIdx.x);
  if (it >= items) return;  // (the whole workgroup)
  Item I = open(it);
  // token row wv of a column tile (1 KiB, one direct-to-LDS instruction) and its eight scales
  auto stage = [&](const Item& J, uint32_t ct, uint8_t* xb, float* xs) {
    if (wv >= J.n) return;
    const uint32_t lane = lane_now();
    const uint32_t t = w8_row(J.tok, wv);
    const __amdgpu_buffer_rsrc_t r = buffer_rsrc(A.x8 + (uint64_t)t * A.cols + (uint64_t)ct * kTileCols, kTileCols);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, AFFX_LDS_PTR(xb + wv * kW8Row), 16, lane * 16u, 0, 0, 0);
    const __amdgpu_buffer_rsrc_t q = buffer_rsrc(A.xs + (uint64_t)t * nkb + ct * 8u, 32u);
    if (lane < 8u) __builtin_amdgcn_raw_ptr_buffer_load_lds(q, AFFX_LDS_PTR(xs + wv * 8u), 4, lane * 4u, 0, 0, 0);
  };
  auto load = [&](Unit& u, const Item& J, uint32_t ct) {
    if (J.rt < nrt) load_unit_ordered(u, J.codes, J.fields, (uint64_t)J.rt * nct + ct, lane_now());
  };

  Unit ua, ub;
  load(ua, I, 0);
  stage(I, 0, xb0, xs0);
  {
    uint32_t cbv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cbv[i] = A.codebook[tid + (uint32_t)i * kW8LT];
    build_lut<kW8KC, kW8LT, 4, true>(lut_s, cbv, tid);
    if (tid < kSegCols / 4) reinterpret_cast<uint32_t*>(zero_s)[tid] = 0u;
  }
  __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
  __syncthreads();

  constexpr int NQ = kW8Light / 4;
  float out[NQ][4] = {};
  uint32_t ct = 0;
  // multiplies the unit by the tile's quads; Q of them (a template of the quad count: no branch
  // between a step's table reads and its MFMAs)
  auto mult = [&](auto qc, Unit& u, const uint8_t* xb, const float* xs) {
    constexpr int Q = decltype(qc)::value;
    const uint32_t lane = lane_now(), c = lane & 15, kg = lane >> 4, copy4 = ((lane >> 1) & (kW8KC - 1)) * 4u;
    v4f acc[Q][2];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q][0] = acc[q][1] = v4f{0.f, 0.f, 0.f, 0.f};
    const uint8_t* src[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint32_t jl = 4u * (uint32_t)q + (c >> 2);
      src[q] = (c & 3u) == kg && jl < I.n ? xb + jl * kW8Row + kg * (uint32_t)kSegCols : zero_s;
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      uint32_t raw[8], bv[2];
      pin_step(u, m);
      lut_lookup_step<kW8KC, true>(u, lut, nullptr, copy4, m, raw, bv);
      const v8i a = lut_finish(raw, bv);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const v8i b = b_step(reinterpret_cast<const u32x4*>(src[q]), m);
        acc[q][m / 4] = mfma(a, b, acc[q][m / 4]);
      }
      asm volatile("" ::: "memory");  // (one step's reads in flight at a time: registers)
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) w8_fold(acc[q][0], acc[q][1], xs + (4u * q + (c >> 2)) * 8u, out[q]);
  };
  // one step, of unit u from buffers (xb, xs), with the next step's going to un and (yb, ys); false after the last
  auto step = [&](Unit& u, Unit& un, const uint8_t* xb, const float* xs, uint8_t* yb, float* ys) -> bool {
    const bool last = ct + 1 == nct;
    const uint32_t itn = last ? seek(it + gridDim.x) : it;
    const bool more = itn < items;
    Item N = I;
    if (last && more) N = open(itn);
    const bool rows_ok = I.rt < nrt;
    const uint32_t lane = lane_now(), c = lane & 15, kg = lane >> 4;
    // (requested here, used after the last column tile's products)
    uint2 rsv = {0u, 0u};
    if (last && rows_ok)
      rsv = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(*AFFX_CONST_PTR(uint64_t, &A.tiles[I.tile].rscales)) +
                                            I.rt * 16u + 4u * kg);
    if (more) {
      load(un, N, last ? 0u : ct + 1u);
      stage(N, last ? 0u : ct + 1u, yb, ys);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (rows_ok) {
      if (I.n > 4u) mult(IConst<2>{}, u, xb, xs);
      else mult(IConst<1>{}, u, xb, xs);
    }
    if (last) {
      if (rows_ok && (c & 3u) == 0u) {
        void* y = reinterpret_cast<void*>(*AFFX_CONST_PTR(uint64_t, &A.tiles[I.tile].y));
        const uint32_t ldt = *AFFX_CONST_PTR(uint32_t, &A.tiles[I.tile].ld), ntt = *AFFX_CONST_PTR(uint32_t, &A.tiles[I.tile].nt);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          if (4u * q + (c >> 2) < I.n) w8_store(A, y, ldt ? ldt : ntt, I.rt * 16u + 4u * kg, 4u * q + (c >> 2), out[q], rsv);
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) out[q][v] = 0.f;
    }
    if (!more) return false;
    it = itn;
    I = N;
    ct = last ? 0u : ct + 1u;
    __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
    __syncthreads();
    return true;
  };
  while (step(ua, ub, xb0, xs0, xb1, xs1) && step(ub, ua, xb1, xs1, xb0, xs0)) {
  }
}

// ---- heavy tiles --------------------------------------------------------------------------------
// Four waves, 64 rows of a tile an item. NQ: the most quads of the launch's tiles; a tile runs the
// passes and quads that its tokens fill. The tokens are staged in passes of at most kW8Pass.
constexpr uint32_t kW8Pass = 32;

template <int NQ>
__global__ void __launch_bounds__(kW8T) w8a8_gemm_kernel(W8a8Args A) {
  constexpr int NP = (4 * NQ + (int)kW8Pass - 1) / (int)kW8Pass;  // passes
  constexpr int QP = NQ / NP;                                        // quads a pass
  AFFX_DYN_LDS(lds);  // xb [4 QP][kW8Row] activation rows of the pass, then xsl [4 x 64] f32 scales
  uint8_t* xb = lds;
  float* xsl = reinterpret_cast<float*>(lds + 4u * QP * kW8Row);
  __shared__ __align__(16) uint32_t lut_s[Lut<kW8KC, true>::kDwords];
  const uint8_t* lut = reinterpret_cast<const uint8_t*>(lut_s);
  // items tile-major, then 64-row blocks
  const uint32_t nrb = (A.rows / kTileRows + kW8Waves - 1) / kW8Waves, items = A.n_tiles * nrb;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t c = lane & 15, kg = lane >> 4, copy4 = ((lane >> 1) & (kW8KC - 1)) * 4u;
  const uint32_t nct = A.cols / kTileCols, nkb = A.cols / 128u;
  auto seek = [&](uint32_t it) -> uint32_t {
    for (; it < items; it += gridDim.x)
      if (w8_tokens(A.tiles, it / nrb, A.cap) > kW8Light) break;
    return it;
  };
  uint32_t it = seek(blockIdx.x);
  if (it >= items) return;  // (the whole workgroup)
  {
    uint32_t cbv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cbv[i] = A.codebook[tid + (uint32_t)i * kW8T];
    build_lut<kW8KC, kW8T, 8, true>(lut_s, cbv, tid);
  }
  const __amdgpu_buffer_rsrc_t xs_r = buffer_rsrc(A.xs, 0x7FFFFFF0u);

  for (; it < items; it = seek(it + gridDim.x)) {
    const uint32_t tile = it / nrb, rb = it - tile * nrb;
    const affx_expert_tile* T = A.tiles + tile;
    const uint32_t ntok = w8_tokens(A.tiles, tile, A.cap);
    const uint32_t rt = rb * kW8Waves + wv;
    const bool rows_ok = rt * kTileRows < A.rows;
    const uint32_t* tok = reinterpret_cast<const uint32_t*>(*AFFX_CONST_PTR(uint64_t, &T->tok));
    const uint8_t* codes = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->codes));
    const uint8_t* fields = reinterpret_cast<const uint8_t*>(*AFFX_CONST_PTR(uint64_t, &T->fields));
    // the lane's four accumulator rows' scales
    uint2 rsv = {0u, 0u};
    if (rows_ok)
      rsv = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(*AFFX_CONST_PTR(uint64_t, &T->rscales)) +
                                            rt * 16u + 4u * kg);
    // the lane's scale dword of each pass (token pass * 4 QP + d / 8, block 8 ct + d % 8 for
    // d = 64 wave + lane; past the pass's tokens: out of the buffer's range, zero)
    uint32_t xs_off[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t d = 64u * wv + lane, jj = (uint32_t)p * 4u * QP + d / 8u;
      xs_off[p] = (d < 32u * QP && jj < ntok) ? ((tok ? tok[jj] : jj) * nkb + d % 8u) * 4u : 0x7FFFFFF0u;
    }

    float out[NQ][4];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) out[q][v] = 0.f;

    // a pass's LDS: the pass's token rows, QP per wave at most (1 KiB each, one direct-to-LDS load
    // instruction), and one scale instruction per wave
    auto stage = [&](int p, uint32_t ct) {
#pragma unroll
      for (int i = 0; i < QP; ++i) {
        const uint32_t jl = wv + 4u * (uint32_t)i, j = (uint32_t)p * 4u * QP + jl;
        if (j >= ntok) break;  // (rows past the tile's tokens are not read)
        const __amdgpu_buffer_rsrc_t r =
            buffer_rsrc(A.x8 + (uint64_t)w8_row(tok, j) * A.cols + (uint64_t)ct * kTileCols, kTileCols);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, AFFX_LDS_PTR(xb + jl * kW8Row), 16, lane * 16u, 0, 0, 0);
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xs_r, AFFX_LDS_PTR(xsl + 64u * wv), 4, xs_off[p] + ct * 32u, 0, 0, 0);
    };

    for (uint32_t ct = 0; ct < nct; ++ct) {
      // this wave's unit of the column tile first (loads complete in issue order)
      Unit u;
      load_unit_ordered(u, codes, fields, (uint64_t)(rows_ok ? rt : 0u) * nct + ct, lane);
      v8i a[8];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        if ((uint32_t)p * 4u * QP >= ntok) break;  // (the same for the whole workgroup)
        __syncthreads();  // the previous pass's reads of the LDS are done
        stage(p, ct);
        if (p == 0) {
          // the wave tile's eight A fragments, while the pass's rows arrive
#pragma unroll
          for (int m = 0; m < 8; ++m) {
            uint32_t raw[8], bv[2];
            pin_step(u, m);
            lut_lookup_step<kW8KC, true>(u, lut, nullptr, copy4, m, raw, bv);
            a[m] = lut_finish(raw, bv);
            asm volatile("" ::: "memory");  // one step's table reads in flight at a time (registers)
          }
        }
        __builtin_amdgcn_s_waitcnt(AFFX_VMCNT(0));
        __syncthreads();
        if (!rows_ok) continue;
#pragma unroll
        for (int ql = 0; ql < QP; ++ql) {
          const int q = p * QP + ql;
          if (4u * (uint32_t)q >= ntok) break;
          const uint32_t jl = 4u * (uint32_t)ql + (c >> 2);
          const bool live = (c & 3u) == kg && (uint32_t)p * 4u * QP + jl < ntok;
          const uint8_t* bsrc = xb + jl * kW8Row + kg * (uint32_t)kSegCols;
          v4f acc0 = v4f{0.f, 0.f, 0.f, 0.f}, acc1 = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int m = 0; m < 8; ++m) {
            v8i b = v8i{0, 0, 0, 0, 0, 0, 0, 0};
            if (live) b = b_step(reinterpret_cast<const u32x4*>(bsrc), m);
            if (m < 4)
              acc0 = mfma(a[m], b, acc0);
            else
              acc1 = mfma(a[m], b, acc1);
          }
          w8_fold(acc0, acc1, xsl + jl * 8u, out[q]);
          // one quad at a time: the next quad's B reads are not hoisted over this one's MFMAs (a
          // compiler memory barrier; the registers of every quad's operands at once would cut the
          // waves a SIMD holds to one)
#pragma unroll
          for (int v = 0; v < 4; ++v) AFFX_PIN(out[q][v]);
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (!rows_ok || (c & 3u) != 0u) continue;
    void* y = reinterpret_cast<void*>(*AFFX_CONST_PTR(uint64_t, &T->y));
    const uint32_t ldt = *AFFX_CONST_PTR(uint32_t, &T->ld), ld = ldt ? ldt : *AFFX_CONST_PTR(uint32_t, &T->nt);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const uint32_t j = 4u * q + (c >> 2);
      if (j < ntok) w8_store(A, y, ld, rt * 16u + 4u * kg, j, out[q], rsv);
    }
  }
}

}  // namespace affx

using namespace affx;

namespace {

// persistent grids: as many workgroups as the device holds at once (two a CU in either kernel)
template <int NQ>
int w8a8_launch(const W8a8Args& A, uint32_t grid, hipStream_t s) {
  constexpr int NP = (4 * NQ + (int)kW8Pass - 1) / (int)kW8Pass, QP = NQ / NP;
  const uint32_t lds = 4u * QP * kW8Row + 4u * 64u * 4u;
  int rc = check_hip(hipFuncSetAttribute((const void*)w8a8_gemm_kernel<NQ>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)lds),
                     "hipFuncSetAttribute(w8a8)");
  if (rc) return rc;
  hipLaunchKernelGGL((w8a8_gemm_kernel<NQ>), dim3(grid), dim3(kW8T), lds, s, A);
  return check_launch("w8a8_gemm_kernel");
}

}  // namespace

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
  hipStream_t s = (hipStream_t)stream;
  A.n_tiles = n_tiles;
  const uint32_t nq = (max_nt + 3u) / 4u;
  A.cap = nq <= 1 ? 4u : nq <= 2 ? 8u : nq <= 4 ? 16u : nq <= 8 ? 32u : 64u;
  int dev = 0, cus = 0, rc;
  if ((rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) ||
      (rc = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute")))
    return rc;
  auto grid = [&](uint32_t waves) {
    const uint64_t items = (uint64_t)n_tiles * ((rows / kTileRows + waves - 1) / waves), most = 2ull * (uint32_t)(cus > 0 ? cus : 1);
    return (uint32_t)(items < most ? items : most);
  };
  // the heavy tiles first: their items are the longer ones
  if (A.cap > kW8Light) {
    const uint32_t g = grid(kW8Waves);
    rc = nq <= 4 ? w8a8_launch<4>(A, g, s) : nq <= 8 ? w8a8_launch<8>(A, g, s) : w8a8_launch<16>(A, g, s);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(w8a8_light_kernel, dim3(grid(kW8LWaves)), dim3(kW8LT), 0, s, A);
  return check_launch("w8a8_light_kernel");
}
