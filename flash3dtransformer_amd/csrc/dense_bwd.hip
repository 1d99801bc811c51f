// Backward of the dense layers for gfx950: weight / bias gradient of a linear layer, LayerNorm backward and the
// backward of the gated activation.  The input gradient of a linear layer is itself a linear layer (dx = dy · w), so it
// runs on the forward kernels with the transposed weight.
//
// The reference takes these from torch.nn.Linear / TransformerEngine autograd (flash3dxfmr/layers/buck_swin.py:159-163,
// elem_wise.py:22-26, stage.py:94-99); nothing of it lives in the reference's own sources.
//
// Weight gradient  dw[n][k] = sum_m dy[m][n] x[m][k]  (fp32 out, bf16 in):
//   the reduction runs over the rows, which is the slow axis of both operands in memory, so both MFMA operands are
//   read TRANSPOSED from LDS (ds_read_b64_tr_b16: a lane receives four consecutive rows of one column).  A workgroup of
//   eight waves (two per SIMD) owns a tile of dw, as wide in either direction as its columns (32, 64, 128 or 256), and one
//   slab of rows; a wave holds up to 64 x 128 of it in accumulator registers and skips the 32 x 32 blocks that lie outside dw.
//   Stages of 32 (256 x 256) to 256 rows (32 x 32), 24 to 40 KB each, stream HBM -> LDS directly (global_load ... lds,
//   no registers) through four stage buffers, so three stages are in flight behind the one being multiplied; one barrier per
//   stage.  Where a tile has fewer blocks than waves, the waves share the rows of a stage and add their sums at the end.
//   Slabs are sized so that the launch is one round of the chip; every slab writes its partial tile to the workspace and a second
//   kernel sums the slabs in a fixed order (no atomics: the result does not depend on scheduling).  The bias gradient rides
//   along in the waves of the first k-tile as one more product with a matrix of ones.
//   What bounds it: the rows' way in.  In tiles of 256 x 256 alone, a 32 x 32 gradient moved 4 KB a stage (12 KB a CU in flight) and
//   fetched seven of eight pieces twice; slabs of consecutive rows made the chip read 256 runs of rows megabytes apart.
//   Both kernels of a call, operands not in any cache, before -> now: 482,304 rows 32 x 32 47.6 -> 29.9 us, 96 x 32 61 -> 51,
//   32 x 128 70 -> 61, 256 x 32 117 -> 101; 241,152 rows 64 x 64 37 -> 30, 512 x 64 118 -> 110; 120,832 rows 1024 x 128 121 -> 115;
//   5,000 rows 64 x 256 19 -> 14; 30,208 rows 4096 x 512 177 (0.71 PFLOP/s) either way.  Errors against fp64 equal or smaller
//   (2.8e-7 -> 1.4e-7 of a 32 x 32 gradient).
#include <algorithm>

#include "f3d_device.h"
#include "f3d_internal.h"

namespace f3d {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

constexpr int kXcd = 8;
constexpr int kWgThreads = 512, kWgWaves = kWgThreads / kWave;
constexpr int kWgNBuf = 4;                   // stage buffers: three stages in flight behind the one being multiplied

// rows of a stage of wn + wk columns: 24 to 40 KB
constexpr int wg_stage_rows(int wn, int wk) {
  const int row = 2 * (wn + wk);
  return row * 256 <= 40960 ? 256 : row * 128 <= 40960 ? 128 : row * 64 <= 40960 ? 64 : 32;
}
// A workgroup's tile of dw: WN x WK columns of dy and x (32, 64, 128 or 256 each), MT rows a stage
template <int WN, int WK>
struct WgGeom {
  static constexpr int ROW = 2 * (WN + WK);                       // bytes of a row of both operands
  static constexpr int MT = wg_stage_rows(WN, WK);
  static constexpr int RA = 2 * WN, RB = 2 * WK;                  // bytes of an LDS row, no padding
  static constexpr int TILE_A = MT * RA, STAGE = MT * ROW, LDS = kWgNBuf * STAGE;
  static constexpr int DMA_A = TILE_A / 1024, DMA = STAGE / 1024;             // direct loads (1 KB each) of a stage
  static constexpr int DMA_WAVE = (DMA + kWgWaves - 1) / kWgWaves;            // ... of a wave (a last one may repeat)
  // the eight waves: over the 32-column blocks of dy, then those of x, what is left of them over the rows of a stage
  static constexpr int NB = WN / 32, KB = WK / 32;
  static constexpr int GN = NB < 4 ? NB : 4, GK = KB < 8 / GN ? KB : 8 / GN, GR = 8 / (GN * GK);
  static constexpr int NI = NB / GN, NJ = KB / GK;                // blocks of a wave
  static constexpr int KS = MT / 16 / GR;                         // k-steps of a wave and stage
};
static_assert(WgGeom<256, 256>::LDS == 128 * 1024 && WgGeom<128, 32>::LDS == 160 * 1024, "stage geometry");

// 16 bytes per lane from global memory straight into LDS: lane l of the wave lands at lds + 16 l
__device__ __forceinline__ void wg_dma16(const void* gbase, uint32_t voff, const char* lds) {
  const uint32_t lds_addr =
      __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)lds);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(gbase)
               : "memory", "m0");
}

// two transposing reads -> one 8-value MFMA operand: slots 0..3 = rows r .. r+3, slots 4..7 = rows r+4 .. r+7 of the
// lane's column (the same row order for both operands, so the products pair up)
template <int ROWB>
__device__ __forceinline__ bf16x8_t read_tr8(const char* p) {
  const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)p);
  const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(p + 4 * ROWB));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// LDS layout of an operand tile: row r at r ROWB, its 16-byte piece c stored at position c ^ wg_swizzle(r).  The
// direct loads write positions linearly (a lane picks the global piece that belongs at its position).  A transposing
// read has 32 lanes touch 64 bytes of each of four consecutive rows; the swizzle sends the four rows to the four
// 64-byte quarters of the 256 bytes the 64 banks serve per clock (without it rows a multiple of 256 bytes apart would all
// meet in the same banks; rows of 128 bytes two by two; rows of 64 bytes need none).
template <int ROWB>
__device__ __forceinline__ uint32_t wg_swizzle(uint32_t r) {
  return ROWB >= 256 ? (r & 3u) << 2 : ROWB == 128 ? ((r >> 1) & 1u) << 2 : 0u;
}

// A slab's rows are every slabs-th stage of the whole: at any time the chip reads one run of rows, not 256 runs that start
// megabytes apart.
template <int WN, int WK>
__global__ __launch_bounds__(kWgThreads) void linear_wgrad_kernel(
    const uint16_t* __restrict__ dy, uint32_t lddy, const uint16_t* __restrict__ x, uint32_t ldx,
    float* __restrict__ part_w, float* __restrict__ part_b, uint32_t M, uint32_t N, uint32_t K, uint32_t n_tiles,
    uint32_t k_tiles, uint32_t slabs, uint32_t items_per_xcd) {
  using G = WgGeom<WN, WK>;
  constexpr int MT = G::MT, RA = G::RA, RB = G::RB, NI = G::NI, NJ = G::NJ, KS = G::KS;
  extern __shared__ __attribute__((aligned(16))) char lds_wg[];
  // workgroups of one XCD take consecutive items, so the tiles of one slab (which re-read the same rows of x and
  // dy) meet in one L2
  const uint32_t tiles = n_tiles * k_tiles, n_items = tiles * slabs;
  const uint32_t item = (blockIdx.x % kXcd) * items_per_xcd + blockIdx.x / kXcd;
  if (blockIdx.x / kXcd >= items_per_xcd || item >= n_items) return;
  const uint32_t slab = item / tiles, tile = item % tiles;
  const uint32_t n0 = (tile / k_tiles) * WN, k0 = (tile % k_tiles) * WK;
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t nw = wave % G::GN, kw = wave / G::GN % G::GK, rw = wave / (G::GN * G::GK);
  const bool with_bias = part_b != nullptr && k0 == 0 && kw == 0;
  // 32 x 32 blocks of this wave that lie inside dw
  const uint32_t n_w = n0 + nw * 32u * NI, k_w = k0 + kw * 32u * NJ;
  const uint32_t ni = n_w >= N ? 0u : min((uint32_t)NI, (N - n_w + 31u) / 32u), nj = k_w >= K ? 0u : min((uint32_t)NJ, (K - k_w + 31u) / 32u);

  // ---- direct loads: load q of a stage fills 1 KB of LDS, the tile of dy first; this wave issues q = wave + 8 i.
  //      Pieces beyond the last column are clamped to the last valid piece (they only reach blocks of dw that are
  //      never stored), rows beyond the last to it (and zeroed in LDS once they have landed). ----
  const uint32_t pieces_a = min((uint32_t)RA / 16u, (N - n0) / 8u), pieces_b = min((uint32_t)RB / 16u, (K - k0) / 8u);
  // (wave < 8: which operand load i belongs to is known at compile time but for one i at most)
  auto dma = [&](int i) { return G::DMA % kWgWaves == 0 ? wave + 8u * i : min(wave + 8u * i, (uint32_t)G::DMA - 1u); };
  auto of_dy = [&](int i) { return 8 * i + 7 < G::DMA_A || (8 * i < G::DMA_A && wave + 8u * i < (uint32_t)G::DMA_A); };
  uint32_t d_row[G::DMA_WAVE], d_col[G::DMA_WAVE];
#pragma unroll
  for (int i = 0; i < G::DMA_WAVE; ++i) {
    const uint32_t q = dma(i);
    const bool a = of_dy(i);
    const uint32_t at = (a ? q : q - G::DMA_A) * 1024u + lane * 16u;
    const uint32_t row = at / (a ? (uint32_t)RA : (uint32_t)RB), pos = at % (a ? (uint32_t)RA : (uint32_t)RB) / 16u;
    const uint32_t c = pos ^ (a ? wg_swizzle<RA>(row) : wg_swizzle<RB>(row));
    d_row[i] = row;
    d_col[i] = min(c, (a ? pieces_a : pieces_b) - 1u) * 16u;
  }
  auto first_row = [&](uint32_t st) { return (st * slabs + slab) * MT; };
  auto issue = [&](uint32_t st) {
    const uint32_t m0 = first_row(st), last = M - 1u - m0;   // m0 < M
    const char* ga = reinterpret_cast<const char*>(dy + (size_t)m0 * lddy + n0);
    const char* gb = reinterpret_cast<const char*>(x + (size_t)m0 * ldx + k0);
    char* buf = lds_wg + (st % kWgNBuf) * G::STAGE;
#pragma unroll
    for (int i = 0; i < G::DMA_WAVE; ++i) {
      const bool a = of_dy(i);      // uniform
      wg_dma16(a ? ga : gb, min(d_row[i], last) * (a ? lddy : ldx) * 2u + d_col[i], buf + dma(i) * 1024);
    }
  };

  // ---- the lane's place in a transposing read: lane p of a 16-lane block points at row p / 4, columns 4 (p % 4)..;
  //      the swizzle value of row p / 4 is that of every row the lane ever reads (they differ by multiples of 4) ----
  const uint32_t half = lane >> 5, p16 = lane & 15u, cgrp = (lane >> 4) & 1u, r0 = 8u * half + p16 / 4u, in_piece = 8u * (p16 & 1u);
  uint32_t a_off[NI], b_off[NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    a_off[i] = r0 * RA + ((((nw * NI + i) * 4u + 2u * cgrp + ((p16 & 3u) >> 1)) ^ wg_swizzle<RA>(r0)) << 4) + in_piece;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    b_off[j] = G::TILE_A + r0 * RB + ((((kw * NJ + j) * 4u + 2u * cgrp + ((p16 & 3u) >> 1)) ^ wg_swizzle<RB>(r0)) << 4) + in_piece;

  f32x16_t acc[NI][NJ], accb[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) accb[i][e] = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  }
  bf16x8_t ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;

  const uint32_t all_stages = (M + MT - 1) / MT;
  const uint32_t n_stage = all_stages > slab ? (all_stages - slab + slabs - 1) / slabs : 0u;
  // waits until this wave's loads of stage st have landed (at most the loads of the later stages, two of them at
  // that point, stay outstanding), zeroes the rows past the slab, and meets the other waves: after the barrier the
  // whole stage is in LDS and every wave has its operands of the stages before it in registers
  auto stage_ready = [&](uint32_t st) {
    const uint32_t later = min(n_stage - 1u - st, 2u);
    if (later == 2u) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * G::DMA_WAVE) : "memory");
    else if (later == 1u) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::DMA_WAVE) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t rows_left = M - first_row(st);
    if (rows_left < (uint32_t)MT) {
      char* buf = lds_wg + (st % kWgNBuf) * G::STAGE;
#pragma unroll
      for (int i = 0; i < G::DMA_WAVE; ++i)
        if (d_row[i] >= rows_left)
          *reinterpret_cast<u32x4_t*>(buf + dma(i) * 1024u + lane * 16u) = u32x4_t{0u, 0u, 0u, 0u};
    }
    wg_barrier_lds();
  };
  bf16x8_t fa[2][NI], fb[2][NJ];
  // k-step ks of this wave: rows 16 (GR ks + rw) .. of the stage
  auto frags = [&](uint32_t st, int ks, bf16x8_t (&a)[NI], bf16x8_t (&b)[NJ]) {
    const char* buf = lds_wg + (st % kWgNBuf) * G::STAGE;
    const uint32_t row = 16u * (G::GR * ks + rw);
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if ((uint32_t)i < ni) a[i] = read_tr8<RA>(buf + a_off[i] + row * RA);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if ((uint32_t)j < nj) b[j] = read_tr8<RB>(buf + b_off[j] + row * RB);
  };
  auto products = [&](const bf16x8_t (&a)[NI], const bf16x8_t (&b)[NJ]) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)i < ni && (uint32_t)j < nj)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    if (with_bias) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if ((uint32_t)i < ni) accb[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], ones, accb[i], 0, 0, 0);
    }
  };
  // Three stages are requested ahead.  The hand-over to the next stage (wait, barrier, first operand reads) sits
  // in front of the last k-step's products of a stage, which run over it.
#pragma unroll
  for (int st = 0; st < kWgNBuf - 1; ++st)
    if ((uint32_t)st < n_stage) issue(st);
  if (n_stage) {
    stage_ready(0);
    frags(0, 0, fa[0], fb[0]);
  }
  static_assert(KS % 2 == 0, "operands of k-step 0 are in the first buffer");
  for (uint32_t st = 0; st < n_stage; ++st) {
    // the buffer of stage st - 1 is free: every wave read the last of it before the barrier that made stage st ready
    if (st + kWgNBuf - 1 < n_stage) issue(st + kWgNBuf - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) {
        frags(st, ks + 1, fa[(ks + 1) & 1], fb[(ks + 1) & 1]);
      } else if (st + 1 < n_stage) {
        stage_ready(st + 1);   // stages st + 2 and st + 3 are the ones still in flight
        frags(st + 1, 0, fa[0], fb[0]);
      }
      products(fa[ks & 1], fb[ks & 1]);
    }
  }

  // ---- waves that shared the rows of a stage: their sums are added in ascending order of the row group ----
  if constexpr (G::GR > 1) {
    __syncthreads();      // the stage buffers are free
    constexpr uint32_t WAVE_B = (NI * NJ + NI) * 4096;
    static_assert((G::GR - 1) * G::GN * G::GK * WAVE_B <= G::LDS, "the waves' sums fit the stage buffers");
    float* const mine = reinterpret_cast<float*>(lds_wg + (wave - G::GN * G::GK) * WAVE_B);
    if (rw > 0) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j <= NJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) mine[((i * (NJ + 1) + j) * 16 + e) * 64 + lane] = j < NJ ? acc[i][j < NJ ? j : 0][e] : accb[i][e];
    }
    __syncthreads();
    if (rw > 0) return;
#pragma unroll 1
    for (uint32_t r = 1; r < (uint32_t)G::GR; ++r) {
      const float* theirs = reinterpret_cast<const float*>(lds_wg + ((r - 1) * G::GN * G::GK + wave) * WAVE_B);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j <= NJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float v = theirs[((i * (NJ + 1) + j) * 16 + e) * 64 + lane];
            if (j < NJ) acc[i][j < NJ ? j : 0][e] += v;
            else accb[i][e] += v;
          }
    }
  }

  // ---- this slab's partial tile: accumulator slot e of a lane is row 8 (e / 4) + 4 half + e % 4, column lane % 32 ----
  float* pw = part_w + (size_t)slab * N * K;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const uint32_t n = n_w + 32u * i + 8u * (e / 4) + 4u * half + (e % 4);
      if (n >= N) continue;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint32_t k = k_w + 32u * j + (lane & 31u);
        if (k < K) pw[(size_t)n * K + k] = acc[i][j][e];
      }
      // every column of the product with the matrix of ones holds the row sum
      if (with_bias && (lane & 31u) == 0) part_b[(size_t)slab * N + n] = accb[i][e];
    }
  }
}

// out[i] = (accumulate ? out[i] : 0) + sum over p of part[p][i], for two arrays in one launch (the weight gradient and,
// in the workgroups past blocks_a, the bias gradient; len_b may be 0).  A workgroup owns 4 LANES consecutive elements
// (lengths are multiples of 4); its 16 partial groups each sum every 16th partial, BATCH 16-byte loads at a time (one at a
// time every partial waited for memory), then the first group adds the group sums in
// ascending order: one fixed summation tree for every LANES.  Many partials (small gradients, 128 to 256 slabs) take 16
// lanes, so that 32 x 32 elements still occupy 16 workgroups: 6.1 -> 4.8 us.  (64 groups of 16 lanes took as long, and their
// longer last sum raised the error of a bias gradient from 1.0e-7 to 1.9e-7 at 482,304 rows.)
template <int LANES, uint32_t BATCH>
__global__ __launch_bounds__(16 * LANES) void sum_partials_kernel(const float* __restrict__ part_a, size_t len_a,
                                                                  float* __restrict__ out_a, uint32_t blocks_a,
                                                                  const float* __restrict__ part_b, size_t len_b,
                                                                  float* __restrict__ out_b, uint32_t n_part,
                                                                  uint32_t accumulate) {
  constexpr uint32_t GROUPS = 16u;
  __shared__ float4 s_sum[GROUPS][LANES];
  const bool second = blockIdx.x >= blocks_a;
  const float* part = second ? part_b : part_a;
  float* out = second ? out_b : out_a;
  const size_t len = second ? len_b : len_a;
  const uint32_t tid = threadIdx.x, l = tid % LANES, g = tid / LANES;
  const size_t i = ((size_t)(blockIdx.x - (second ? blocks_a : 0u)) * LANES + l) * 4u;
  float4 s = {0.f, 0.f, 0.f, 0.f};
  if (n_part <= GROUPS) {      // uniform
    if (i < len && g < n_part) s = *reinterpret_cast<const float4*>(part + (size_t)g * len + i);
  } else if (i < len) {
    for (uint32_t p = g; p < n_part; p += BATCH * GROUPS) {
      float4 v[BATCH];
#pragma unroll
      for (uint32_t u = 0; u < BATCH; ++u) {
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p + u * GROUPS < n_part) v[u] = *reinterpret_cast<const float4*>(part + (size_t)(p + u * GROUPS) * len + i);
      }
#pragma unroll
      for (uint32_t u = 0; u < BATCH; ++u) { s.x += v[u].x; s.y += v[u].y; s.z += v[u].z; s.w += v[u].w; }
    }
  }
  s_sum[g][l] = s;
  __syncthreads();
  if (g == 0 && i < len) {
    float4 t = {0.f, 0.f, 0.f, 0.f};
    if (accumulate) t = *reinterpret_cast<const float4*>(out + i);
#pragma unroll
    for (uint32_t r = 0; r < GROUPS; ++r) {
      const float4 v = s_sum[r][l];
      t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
    }
    *reinterpret_cast<float4*>(out + i) = t;
  }
}

// ---- LayerNorm backward: LPR lanes per row, 8 channels per lane.
//   xhat = (x - mean) rstd, g = dh gamma, dx = rstd (g - mean(g) - xhat mean(g xhat)) (+ dres),
//   dgamma = sum_rows dh xhat, dbeta = sum_rows dh.  A thread walks rows with a grid stride and keeps its 8 + 8 column
//   sums in registers; the workgroup combines them through LDS and writes one partial per workgroup.
//   APART: dx is rounded to bf16 before dres is added, as two tensors added afterwards would be (the bits of that sum, without
//   writing dx and reading both again: 14 additions of 19 us in a training step of 482,304 rows). ----
template <int LPR, bool APART>
__global__ __launch_bounds__(256) void layernorm_bwd_kernel(const uint16_t* __restrict__ x, uint32_t ldx,
                                                            const uint16_t* dh, uint32_t lddh,
                                                            const uint16_t* __restrict__ gamma,
                                                            const uint16_t* dres, uint32_t lddr,
                                                            uint16_t* dx, uint32_t lddx,
                                                            float* __restrict__ part, uint32_t M, float eps) {
  constexpr int C = LPR * 8, RPB = 256 / LPR;
  __shared__ float s_col[256][17];
  const uint32_t tid = threadIdx.x, sub = tid % LPR, slot = tid / LPR;
  float g8[8], dg[8], db[8];
  {
    const u32x4_t g = *reinterpret_cast<const u32x4_t*>(gamma + sub * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) { g8[2 * e] = bf16_lo(g[e]); g8[2 * e + 1] = bf16_hi(g[e]); }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) dg[e] = db[e] = 0.f;
  // every lane of a row group runs the same number of iterations (the shuffles need all of them)
  for (uint32_t base = blockIdx.x * RPB; base < M; base += gridDim.x * RPB) {
    const uint32_t row = base + slot;
    const bool ok = row < M;
    u32x4_t vx = {0u, 0u, 0u, 0u}, vd = {0u, 0u, 0u, 0u}, vr = {0u, 0u, 0u, 0u};
    if (ok) {
      vx = *reinterpret_cast<const u32x4_t*>(x + (size_t)row * ldx + sub * 8);
      vd = *reinterpret_cast<const u32x4_t*>(dh + (size_t)row * lddh + sub * 8);
      if (dres) vr = *reinterpret_cast<const u32x4_t*>(dres + (size_t)row * lddr + sub * 8);
    }
    float xv[8], dv[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xv[2 * e] = bf16_lo(vx[e]); xv[2 * e + 1] = bf16_hi(vx[e]);
      dv[2 * e] = bf16_lo(vd[e]); dv[2 * e + 1] = bf16_hi(vd[e]);
    }
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) sum += xv[e];
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
    const float mean = sum / (float)C;
    float sq = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { xv[e] -= mean; sq += xv[e] * xv[e]; }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) sq += __shfl_xor(sq, off, kWave);
    const float rstd = rsqrtf(sq / (float)C + eps);
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      xv[e] *= rstd;                       // xhat
      const float g = dv[e] * g8[e];
      s1 += g; s2 += g * xv[e];
      dg[e] += dv[e] * xv[e]; db[e] += dv[e];   // rows past the end contribute zeros (dh = 0)
    }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) {
      s1 += __shfl_xor(s1, off, kWave);
      s2 += __shfl_xor(s2, off, kWave);
    }
    s1 /= (float)C; s2 /= (float)C;
    if (ok) {
      u32x4_t t;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (APART) {
          const uint32_t own = pack_bf16x2(rstd * (dv[2 * e] * g8[2 * e] - s1 - xv[2 * e] * s2),
                                           rstd * (dv[2 * e + 1] * g8[2 * e + 1] - s1 - xv[2 * e + 1] * s2));
          t[e] = pack_bf16x2(bf16_lo(own) + bf16_lo(vr[e]), bf16_hi(own) + bf16_hi(vr[e]));
        } else {
          float f0 = rstd * (dv[2 * e] * g8[2 * e] - s1 - xv[2 * e] * s2) + bf16_lo(vr[e]);
          float f1 = rstd * (dv[2 * e + 1] * g8[2 * e + 1] - s1 - xv[2 * e + 1] * s2) + bf16_hi(vr[e]);
          t[e] = pack_bf16x2(f0, f1);
        }
      }
      *reinterpret_cast<u32x4_t*>(dx + (size_t)row * lddx + sub * 8) = t;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) { s_col[tid][e] = dg[e]; s_col[tid][8 + e] = db[e]; }
  __syncthreads();
  // thread (sub, e) for e < 16 sums the RPB row slots of its column
  for (uint32_t o = tid; o < LPR * 16u; o += 256u) {
    const uint32_t su = o / 16u, e = o % 16u;
    float s = 0.f;
    for (uint32_t r = 0; r < (uint32_t)RPB; ++r) s += s_col[r * LPR + su][e];
    // partial layout per workgroup: dgamma [C] then dbeta [C]
    part[(size_t)blockIdx.x * 2u * C + (e / 8u) * C + su * 8u + (e % 8u)] = s;
  }
}

// ---- gated activation backward: a = silu(z1) z2, dz1 = da z2 s (1 + z1 (1 - s)), dz2 = da silu(z1), s = sigmoid(z1);
//      z = [z1 | z2] per row.  dz may alias z and a may alias da (a thread reads its pieces before it writes them). ----
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const uint16_t* z, uint32_t ldz, const uint16_t* da,
                                                         uint32_t ldda, uint16_t* dz, uint32_t lddz, uint16_t* a,
                                                         uint32_t lda, uint32_t M, uint32_t H) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t cpr = H / 8;
  const uint32_t row = (uint32_t)(gid / cpr), ch = (uint32_t)(gid % cpr) * 8;
  if (row >= M) return;
  const u32x4_t v1 = *reinterpret_cast<const u32x4_t*>(z + (size_t)row * ldz + ch);
  const u32x4_t v2 = *reinterpret_cast<const u32x4_t*>(z + (size_t)row * ldz + H + ch);
  const u32x4_t vd = *reinterpret_cast<const u32x4_t*>(da + (size_t)row * ldda + ch);
  u32x4_t o1, o2, oa;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float r1[2], r2[2], ra[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float z1 = h ? bf16_hi(v1[e]) : bf16_lo(v1[e]);
      const float z2 = h ? bf16_hi(v2[e]) : bf16_lo(v2[e]);
      const float d = h ? bf16_hi(vd[e]) : bf16_lo(vd[e]);
      const float s = 1.f / (1.f + __expf(-z1));
      const float sl = z1 * s;
      ra[h] = sl * z2;
      r1[h] = d * z2 * s * (1.f + z1 * (1.f - s));
      r2[h] = d * sl;
    }
    o1[e] = pack_bf16x2(r1[0], r1[1]);
    o2[e] = pack_bf16x2(r2[0], r2[1]);
    oa[e] = pack_bf16x2(ra[0], ra[1]);
  }
  *reinterpret_cast<u32x4_t*>(dz + (size_t)row * lddz + ch) = o1;
  *reinterpret_cast<u32x4_t*>(dz + (size_t)row * lddz + H + ch) = o2;
  if (a) *reinterpret_cast<u32x4_t*>(a + (size_t)row * lda + ch) = oa;
}

// dgamma / dbeta from the per-workgroup partial rows [dgamma | dbeta].  A workgroup owns 16 columns; its 64 row
// groups each sum every 64th partial row, eight loads at a time (2048 rows: 5 to 7 us a launch; one at a time 11.7), then
// one thread per column adds the 64 group sums in ascending order: a fixed summation tree.
__global__ __launch_bounds__(1024) void ln_bwd_reduce_kernel(const float* __restrict__ part, uint32_t n_part, uint32_t C,
                                                             float* __restrict__ dgamma, float* __restrict__ dbeta,
                                                             uint32_t accumulate) {
  __shared__ float s_red[64][17];
  const uint32_t tid = threadIdx.x, col = blockIdx.x * 16u + (tid & 15u), rg = tid >> 4;
  float s = 0.f;
  if (col < 2u * C)
    for (uint32_t p = rg; p < n_part; p += 512u) {
      float v[8];
#pragma unroll
      for (uint32_t u = 0; u < 8u; ++u) v[u] = p + 64u * u < n_part ? part[(size_t)(p + 64u * u) * 2u * C + col] : 0.f;
#pragma unroll
      for (uint32_t u = 0; u < 8u; ++u) s += v[u];
    }
  s_red[rg][tid & 15u] = s;
  __syncthreads();
  if (tid < 16u && col < 2u * C) {
    float* out = col < C ? dgamma + col : dbeta + (col - C);
    float t = accumulate ? *out : 0.f;
#pragma unroll 16
    for (uint32_t r = 0; r < 64u; ++r) t += s_red[r][tid];
    *out = t;
  }
}

int n_cu_of(int device, uint32_t* n_cu) {
  int v = 0;
  F3D_CHECK_HIP(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, device));
  *n_cu = v > 0 ? (uint32_t)v : 256u;
  return F3D_OK;
}

struct WgLaunch {
  const uint16_t *dy, *x;
  uint32_t lddy, ldx, m, n, k, n_tiles, k_tiles, n_cu;
  int device;
  bool bias;
  hipStream_t stream;
  uint32_t slabs;               // out: row slabs, and where their partial tiles lie
  float *part_w, *part_b;
};

template <int WN, int WK>
int launch_wgrad(WgLaunch& l) {
  using G = WgGeom<WN, WK>;
  // one round of the chip: as many row slabs as there are compute units per tile
  const uint32_t tiles = l.n_tiles * l.k_tiles, stages = cdiv_u32(l.m, G::MT);
  l.slabs = tiles >= l.n_cu ? 1u : l.n_cu / tiles;
  if (l.slabs > stages) l.slabs = stages ? stages : 1u;
  const size_t part_w_bytes = (size_t)l.slabs * l.n * l.k * 4, part_b_bytes = l.bias ? (size_t)l.slabs * l.n * 4 : 0;
  char* ws = (char*)workspace(l.device, part_w_bytes + part_b_bytes, l.stream);
  if (!ws) return F3D_ERR_RUNTIME;
  l.part_w = (float*)ws;
  l.part_b = l.bias ? (float*)(ws + part_w_bytes) : nullptr;
  static bool attr_set[64] = {};
  if (l.device >= 0 && l.device < 64 && !attr_set[l.device]) {
    F3D_CHECK_HIP(hipFuncSetAttribute((const void*)linear_wgrad_kernel<WN, WK>, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS));
    attr_set[l.device] = true;
  }
  const uint32_t items_per_xcd = cdiv_u32(tiles * l.slabs, kXcd);
  hipLaunchKernelGGL((linear_wgrad_kernel<WN, WK>), dim3(items_per_xcd * kXcd), dim3(kWgThreads), G::LDS, l.stream, l.dy, l.lddy, l.x,
                     l.ldx, l.part_w, l.part_b, l.m, l.n, l.k, l.n_tiles, l.k_tiles, l.slabs, items_per_xcd);
  return F3D_OK;
}

}  // namespace
}  // namespace f3d

extern "C" {

int f3d_linear_wgrad_bf16(const f3d_bf16_t* dy, uint32_t lddy, const f3d_bf16_t* x, uint32_t ldx, float* dw, float* db,
                          uint32_t m, uint32_t n, uint32_t k, uint32_t accumulate, int device, void* stream) {
  using namespace f3d;
  F3D_CHECK_ARG(((dy && x) || m == 0) && dw, "null tensor pointer");
  F3D_CHECK_ARG(n > 0 && k > 0 && n % 8 == 0 && k % 8 == 0, "n=%u and k=%u must be positive multiples of 8", n, k);
  F3D_CHECK_ARG(lddy >= n && lddy % 8 == 0 && ldx >= k && ldx % 8 == 0,
                "row strides must be multiples of 8 and cover a row (lddy=%u ldx=%u)", lddy, ldx);
  F3D_CHECK_ARG((((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dw | (uintptr_t)db) & 15u) == 0,
                "dy / x / dw / db must be 16-byte aligned");
  DeviceGuard guard(device);
  F3D_CHECK_ARG(guard.ok, "cannot select device %d", device);
  hipStream_t s = (hipStream_t)stream;
  SyncBracket sync(s);
  uint32_t n_cu = 0;
  if (int rc = n_cu_of(device, &n_cu)) return rc;
  // tile of dw per workgroup: the narrowest width that holds all columns, 256 where none does
  auto width = [](uint32_t c) { return c <= 32u ? 32u : c <= 64u ? 64u : c <= 128u ? 128u : 256u; };
  uint32_t wn = width(n), wk = width(k);
  // The direct loads take 32-bit byte offsets from a stage's first row.  Rows so far apart that a tall stage does not fit
  // (8.4 million elements at 256 rows a stage) take the widest tile, whose stages have 32 rows.
  auto reach = [&](uint32_t rows) { return (uint64_t)(std::min(rows, std::max(m, 1u)) - 1u) * std::max(lddy, ldx) * 2u + 512u; };
  if (reach((uint32_t)wg_stage_rows((int)wn, (int)wk)) >> 32) wn = wk = 256u;
  F3D_CHECK_ARG(reach((uint32_t)wg_stage_rows((int)wn, (int)wk)) >> 32 == 0, "rows of %u or %u elements lie too far apart", lddy, ldx);
  const uint32_t n_tiles = cdiv_u32(n, wn), k_tiles = cdiv_u32(k, wk);
  const size_t nk = (size_t)n * k;
  WgLaunch l = {dy, x, lddy, ldx, m, n, k, n_tiles, k_tiles, n_cu, device, db != nullptr, s};
  int rc = F3D_OK;
#define F3D_WG(WN, WK) \
  if (wn == WN && wk == WK) rc = launch_wgrad<WN, WK>(l)
#define F3D_WGS(WN) F3D_WG(WN, 32); F3D_WG(WN, 64); F3D_WG(WN, 128); F3D_WG(WN, 256)
  F3D_WGS(32); F3D_WGS(64); F3D_WGS(128); F3D_WGS(256);
#undef F3D_WGS
#undef F3D_WG
  if (rc != F3D_OK) return rc;
  auto sum = [&](auto kern, uint32_t lanes) {
    const uint32_t per_block = 4 * lanes;
    const uint32_t blocks_w = (uint32_t)((nk + per_block - 1) / per_block), blocks_b = db ? cdiv_u32(n, per_block) : 0u;
    hipLaunchKernelGGL(kern, dim3(blocks_w + blocks_b), dim3(16 * lanes), 0, s, l.part_w, nk, dw, blocks_w,
                       l.part_b, db ? (size_t)n : (size_t)0, db, l.slabs, accumulate);
  };
  if (l.slabs > 64) sum(sum_partials_kernel<16, 16>, 16u);
  else sum(sum_partials_kernel<64, 8>, 64u);
  F3D_CHECK_HIP(hipGetLastError());
  return F3D_OK;
}

static int layernorm_bwd(const f3d_bf16_t* x, uint32_t ldx, const f3d_bf16_t* dh, uint32_t lddh, const f3d_bf16_t* gamma,
                         const f3d_bf16_t* dres, uint32_t lddr, f3d_bf16_t* dx, uint32_t lddx, float* dgamma, float* dbeta,
                         uint32_t m, uint32_t c, float eps, uint32_t accumulate, bool apart, int device, void* stream) {
  using namespace f3d;
  F3D_CHECK_ARG(((x && dh && dx) || m == 0) && gamma && dgamma && dbeta, "null tensor pointer");
  if (!(c == 32 || c == 64 || c == 128 || c == 256 || c == 512)) {
    set_error("No kernel found for LayerNorm backward at width %u (supported: 32, 64, 128, 256, 512)", c);
    return F3D_ERR_UNSUPPORTED;
  }
  F3D_CHECK_ARG(ldx >= c && ldx % 8 == 0 && lddh >= c && lddh % 8 == 0 && lddx >= c && lddx % 8 == 0 &&
                    (!dres || (lddr >= c && lddr % 8 == 0)),
                "row strides must be multiples of 8 and cover a row");
  F3D_CHECK_ARG((((uintptr_t)x | (uintptr_t)dh | (uintptr_t)gamma | (uintptr_t)dres | (uintptr_t)dx) & 15u) == 0,
                "x / dh / gamma / dres / dx must be 16-byte aligned");
  DeviceGuard guard(device);
  F3D_CHECK_ARG(guard.ok, "cannot select device %d", device);
  hipStream_t s = (hipStream_t)stream;
  SyncBracket sync(s);
  uint32_t n_cu = 0;
  if (int rc = n_cu_of(device, &n_cu)) return rc;
  const uint32_t rpb = 256u / (c / 8u);
  uint32_t wgs = cdiv_u32(m, rpb);
  if (wgs > n_cu * 8u) wgs = n_cu * 8u;
  if (wgs == 0) wgs = 1;
  float* part = (float*)workspace(device, (size_t)wgs * 2u * c * 4u, s);
  if (!part) return F3D_ERR_RUNTIME;
#define F3D_LNB(LPR)                                                                                                          \
  if (apart)                                                                                                                 \
    hipLaunchKernelGGL((layernorm_bwd_kernel<LPR, true>), dim3(wgs), dim3(256), 0, s, x, ldx, dh, lddh, gamma, dres, lddr, dx, \
                       lddx, part, m, eps);                                                                                  \
  else                                                                                                                       \
    hipLaunchKernelGGL((layernorm_bwd_kernel<LPR, false>), dim3(wgs), dim3(256), 0, s, x, ldx, dh, lddh, gamma, dres, lddr, dx, \
                       lddx, part, m, eps)
  switch (c) {
    case 32: F3D_LNB(4); break;
    case 64: F3D_LNB(8); break;
    case 128: F3D_LNB(16); break;
    case 256: F3D_LNB(32); break;
    default: F3D_LNB(64); break;
  }
#undef F3D_LNB
  hipLaunchKernelGGL(ln_bwd_reduce_kernel, dim3(cdiv_u32(2u * c, 16)), dim3(1024), 0, s, part, wgs, c, dgamma, dbeta,
                     accumulate);
  F3D_CHECK_HIP(hipGetLastError());
  return F3D_OK;
}

int f3d_layernorm_bwd_bf16(const f3d_bf16_t* x, uint32_t ldx, const f3d_bf16_t* dh, uint32_t lddh,
                           const f3d_bf16_t* gamma, const f3d_bf16_t* dres, uint32_t lddr, f3d_bf16_t* dx, uint32_t lddx,
                           float* dgamma, float* dbeta, uint32_t m, uint32_t c, float eps, uint32_t accumulate,
                           int device, void* stream) {
  return layernorm_bwd(x, ldx, dh, lddh, gamma, dres, lddr, dx, lddx, dgamma, dbeta, m, c, eps, accumulate, false, device, stream);
}

int f3d_layernorm_bwd_add_bf16(const f3d_bf16_t* x, uint32_t ldx, const f3d_bf16_t* dh, uint32_t lddh,
                               const f3d_bf16_t* gamma, const f3d_bf16_t* dres, uint32_t lddr, f3d_bf16_t* dx, uint32_t lddx,
                               float* dgamma, float* dbeta, uint32_t m, uint32_t c, float eps, uint32_t accumulate,
                               int device, void* stream) {
  F3D_CHECK_ARG(dres || m == 0, "null tensor pointer");
  return layernorm_bwd(x, ldx, dh, lddh, gamma, dres, lddr, dx, lddx, dgamma, dbeta, m, c, eps, accumulate, true, device, stream);
}

int f3d_swiglu_bwd_bf16(const f3d_bf16_t* z, uint32_t ldz, const f3d_bf16_t* da, uint32_t ldda, f3d_bf16_t* dz,
                        uint32_t lddz, f3d_bf16_t* a, uint32_t lda, uint32_t m, uint32_t hidden, int device,
                        void* stream) {
  using namespace f3d;
  F3D_CHECK_ARG(z && da && dz, "null tensor pointer");
  F3D_CHECK_ARG(hidden > 0 && hidden % 8 == 0, "hidden=%u must be a positive multiple of 8", hidden);
  F3D_CHECK_ARG(ldz >= 2 * hidden && ldz % 8 == 0 && lddz >= 2 * hidden && lddz % 8 == 0 && ldda >= hidden &&
                    ldda % 8 == 0 && (!a || (lda >= hidden && lda % 8 == 0)),
                "row strides must be multiples of 8 and cover a row");
  F3D_CHECK_ARG((((uintptr_t)z | (uintptr_t)da | (uintptr_t)dz | (uintptr_t)a) & 15u) == 0,
                "z / da / dz / a must be 16-byte aligned");
  if (m == 0) return F3D_OK;
  DeviceGuard guard(device);
  F3D_CHECK_ARG(guard.ok, "cannot select device %d", device);
  hipStream_t s = (hipStream_t)stream;
  SyncBracket sync(s);
  const size_t threads = (size_t)m * (hidden / 8);
  F3D_CHECK_ARG((threads + 255) / 256 <= 0x7FFFFFFFull, "too many rows");
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0, s, z, ldz, da, ldda, dz,
                     lddz, a, lda, m, hidden);
  F3D_CHECK_HIP(hipGetLastError());
  return F3D_OK;
}

}  // extern "C"
