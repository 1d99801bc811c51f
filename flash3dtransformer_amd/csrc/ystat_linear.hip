// Output-panel ("y-stationary") linear layer for gfx950: y = x wT + bias (+ residual) for inner dimensions that the
// row-panel kernel does not take (above all long ones): the fc2 of the blocks' MLPs (flash3dxfmr/layers/elem_wise.py:22-26,
// where the reference runs te.LayerNormMLP's second GEMM) and the input gradients of QKV and fc1.
//
// The row-panel kernel keeps x in registers, which stops at 512 inner features.  Here the OUTPUT is what stays in
// registers: a workgroup of eight waves owns 128 or 256 rows x 64 to 256 output columns; waves w and w + 4 (the two waves
// of a SIMD) share a block of rows and split the columns, so a wave holds at most 64 rows x 128 columns of fp32
// accumulators (128 registers) and two waves per SIMD fit.  Rows of x and of w stream through LDS 64 inner features at a
// time, straight from HBM / L2 (global_load ... lds).  The product is formed transposed (A operand = rows of w) so that a
// lane ends up with 4 consecutive output columns of one row for the epilogue.
//
// What bounds it: a direct load of whole 128-byte pieces moves 64 bytes a clock and CU, one of 32-byte pieces 18 (linear
// loads: 64), measured on L2-resident data.  With x fetched in 32-byte pieces in operand order the loads took twice
// the time of the products; in whole lines with the pieces swizzled they take half of it, w needs no re-laid copy, and
// the matrix cores set the pace.  30,208 x 512, K = 4096: 155 -> 126 us (1.0 PFLOP/s; the tiled GEMM 207), 60,416 x 256,
// K = 1024: 48 -> 40 us, 8,192 x 512, K = 4096: 46 us (tiled GEMM 70), 1,536 x 512, K = 2048: 24 us (37), 20 in 64 columns.
#include "xstat_common.h"
#include <algorithm>

namespace f3d {

// A ring of 2 (256 x 256) to 6 (128 x 64) buffers, each w and x of one chunk.
constexpr int kYsWaves = 8, kYsChunkK = 64;
constexpr uint32_t kYsXcd = 8;

template <int N, int MT>
struct YsGeom {
  static constexpr int ROWS = 128 * MT;                   // rows of a workgroup
  static constexpr int OTW = N / 64;                      // output column tiles per wave
  static constexpr int ROWB = kYsChunkK * 2;              // an LDS row: 64 inner features of one row of x or w
  static constexpr int W_BYTES = N * ROWB, BUF = W_BYTES + ROWS * ROWB;
  static constexpr int NB = 160 * 1024 / BUF;             // chunk buffers
  static constexpr int W_DMA = N / 64, X_DMA = ROWS / 64; // direct loads (8 rows each) per wave and chunk
  static constexpr size_t lds_bytes() { return (size_t)NB * BUF; }
};

__device__ __forceinline__ void ys_wait_vm(uint32_t n) {
  switch (n) {
#define F3D_W(V) case V: __builtin_amdgcn_s_waitcnt(0x0F70 | V); break;
    F3D_W(0) F3D_W(1) F3D_W(2) F3D_W(3) F3D_W(4) F3D_W(5) F3D_W(6) F3D_W(7) F3D_W(8) F3D_W(9) F3D_W(10) F3D_W(11)
    F3D_W(12) F3D_W(13) F3D_W(14) F3D_W(15)
#undef F3D_W
    // counts of 16 and more: the two high bits of the count sit in bits 15:14 of the immediate
#define F3D_W(V) case V: __builtin_amdgcn_s_waitcnt(0x0F70 | (V & 15) | ((V >> 4) << 14)); break;
    F3D_W(16) F3D_W(17) F3D_W(18) F3D_W(19) F3D_W(20) F3D_W(21) F3D_W(22) F3D_W(23) F3D_W(24) F3D_W(25) F3D_W(26)
    F3D_W(27) F3D_W(28) F3D_W(29) F3D_W(30) F3D_W(31)
#undef F3D_W
    default: __builtin_amdgcn_s_waitcnt(0x0F70); break;
  }
}

// A workgroup's panel: 128 MT rows x N of the NT output columns; bias [NT] may be null
template <int N, int MT>
__global__ __launch_bounds__(64 * kYsWaves, 2) void ystat_linear_kernel(
    const uint16_t* __restrict__ x, uint32_t ldx, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
    const uint16_t* __restrict__ residual, uint32_t ldr, uint16_t* __restrict__ y, uint32_t ldy, uint32_t M,
    uint32_t K, uint32_t NT) {
  using G = YsGeom<N, MT>;
  constexpr int WAVES = kYsWaves, NB = G::NB, OTW = G::OTW;
  constexpr int ROWS_WG = G::ROWS;
  extern __shared__ __attribute__((aligned(1024))) char lds_ys[];

  const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const uint32_t lq = lane & 31u, half = lane >> 5;
  const uint32_t rb = wave & 3u, cg = wave >> 2;          // row block of 32 MT rows, half of the panel's columns
  // Workgroups go round the XCDs in launch order.  The column panels of one row panel run on one XCD, whose L2 serves their
  // reads of x after the first, as long as there are eight row panels to share out; the column panels of the last up to
  // seven go to all XCDs (with those on one XCD each, 128 rows x 8,192 outputs, K = 1024, kept 32 CUs busy for two rounds:
  // 27 us, the tiled GEMM 19, now 12.6)
  const uint32_t n_pan = NT / N, whole = gridDim.x / n_pan / kYsXcd * kYsXcd * n_pan, slot = blockIdx.x / kYsXcd;
  const bool grouped = blockIdx.x < whole;
  const uint32_t row_pan = grouped ? slot / n_pan * kYsXcd + blockIdx.x % kYsXcd : blockIdx.x / n_pan;
  const uint32_t wg_row0 = row_pan * ROWS_WG, col0 = (grouped ? slot : blockIdx.x) % n_pan * N;
  const uint32_t row0 = wg_row0 + rb * (32 * MT);

  // accumulators start from the bias: acc[o][mt][g*4+r] <-> output column (cg*OTW + o)*32 + g*8 + half*4 + r, row lq
  f32x16_t acc[OTW][MT];
#pragma unroll
  for (int o = 0; o < OTW; ++o)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint2 bb = {0u, 0u};
      if (bias) bb = *reinterpret_cast<const uint2*>(bias + col0 + (cg * OTW + o) * 32 + g * 8 + half * 4);
      const float b[4] = {bf16_lo(bb.x), bf16_hi(bb.x), bf16_lo(bb.y), bf16_hi(bb.y)};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[o][mt][g * 4 + r] = b[r];
    }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // nothing of this wave is in flight when the direct loads start

  // ---- streaming ----
  const uint32_t nchunk = K / kYsChunkK;
  constexpr uint32_t kPerChunk = G::W_DMA + G::X_DMA;     // direct loads of this wave per chunk
  // A direct load fills rows 8 q .. 8 q + 7 (q = wave + 8 i) with whole 128-byte pieces of their source rows; the
  // 16-byte piece p of row r sits at position p ^ (r / 2) % 8, so that the 16 rows of a quarter of an operand read meet
  // 16 different places of the 256 bytes the banks serve.  Rows past M read row M - 1.
  const uint32_t l_row = lane / 8u, l_piece = ((lane & 7u) ^ ((4u * wave + lane / 16u) & 7u)) * 16u;
  uint32_t x_lane[G::X_DMA];
#pragma unroll
  for (int i = 0; i < G::X_DMA; ++i)
    x_lane[i] = (min(wg_row0 + (wave + 8u * i) * 8u + l_row, M - 1) - wg_row0) * ldx * 2u + l_piece;
  const uint32_t w_lane = l_row * K * 2u + l_piece;
  const char* x_wg = reinterpret_cast<const char*>(x + (size_t)wg_row0 * ldx);
  const char* w_wg = reinterpret_cast<const char*>(w + (size_t)(col0 + wave * 8u) * K);
  auto dma_chunk = [&](uint32_t c) __attribute__((always_inline)) {
    char* buf = lds_ys + (c % NB) * G::BUF;
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)G::W_DMA; ++i)
      xs_lds_dma16(w_wg + ((size_t)i * 64u * K + (size_t)c * kYsChunkK) * 2u, w_lane, buf + (wave + i * WAVES) * 1024);
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)G::X_DMA; ++i)
      xs_lds_dma16(x_wg + (size_t)c * (kYsChunkK * 2), x_lane[i], buf + G::W_BYTES + (wave + i * WAVES) * 1024);
  };
#pragma unroll
  for (uint32_t c = 0; c < NB - 1u; ++c)
    if (c < nchunk) dma_chunk(c);
  // chunk 0 must have landed; the younger chunks may stay in flight
  ys_wait_vm(min(NB - 2u, nchunk - 1u) * kPerChunk);
  wg_barrier_lds();

  const uint32_t piece0 = (half ^ ((lq / 2u) & 7u)) * 16u;      // of k-step 0; k-step s: ^ 32 s
  for (uint32_t ci = 0; ci < nchunk; ++ci) {
    // chunk ci + NB - 1 goes into the buffer of chunk ci - 1, which every wave has left
    if (ci + (NB - 1) < nchunk) dma_chunk(ci + (NB - 1));
    const char* buf = lds_ys + (ci % NB) * G::BUF;
    const char* sx = buf + G::W_BYTES + (rb * MT * 32 + lq) * G::ROWB;
    const char* sw = buf + (cg * OTW * 32 + lq) * G::ROWB;
#pragma unroll
    for (uint32_t s = 0; s < kYsChunkK / 16; ++s) {
      const uint32_t at = piece0 ^ (s * 32u);
      bf16x8_t xb[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xb[mt] = *reinterpret_cast<const bf16x8_t*>(sx + mt * 32 * G::ROWB + at);
#pragma unroll
      for (int o = 0; o < OTW; ++o) {
        const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(sw + o * 32 * G::ROWB + at);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[o][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, xb[mt], acc[o][mt], 0, 0, 0);
      }
    }
    // chunk ci + 1 must have landed: what may stay in flight are the chunks after it that have been requested
    const uint32_t requested = min(ci + (NB - 1), nchunk - 1);     // youngest chunk requested so far
    ys_wait_vm(requested > ci + 1 ? (requested - (ci + 1)) * kPerChunk : 0);
    wg_barrier_lds();   // not __syncthreads(): that would also wait for the chunks that are meant to stay in flight
  }

  // ---- output: bf16 (+ residual), through a wave-private LDS patch so that the stores are row-contiguous.  The
  //      residual pieces of the wave's whole panel are requested first: one memory latency for all of them ----
  static_assert((size_t)WAVES * 32 * kPatchRow * 2 <= G::lds_bytes(), "the output patches alias the chunk buffers");
  uint16_t* patch = reinterpret_cast<uint16_t*>(lds_ys) + wave * (32 * kPatchRow);
  uint16_t* y_wg = y + (size_t)wg_row0 * ldy;
  const uint16_t* res_wg = residual ? residual + (size_t)wg_row0 * ldr : nullptr;
  u32x4_t rres[MT][OTW][2];
  if (residual) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int o = 0; o < OTW; ++o)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
          const uint32_t rr = (lane >> 2) + h2 * 16, ch = (lane & 3u) * 8;
          const uint32_t row = min(row0 + mt * 32 + rr, M - 1);
          rres[mt][o][h2] = *reinterpret_cast<const u32x4_t*>(res_wg + ((row - wg_row0) * ldr + col0 + (cg * OTW + o) * 32 + ch));
        }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int o = 0; o < OTW; ++o) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint2 pk;   // a Linear's output is bf16
        pk.x = pack_bf16x2(acc[o][mt][g * 4 + 0], acc[o][mt][g * 4 + 1]);
        pk.y = pack_bf16x2(acc[o][mt][g * 4 + 2], acc[o][mt][g * 4 + 3]);
        *reinterpret_cast<uint2*>(patch + lq * kPatchRow + g * 8 + half * 4) = pk;
      }
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        const uint32_t rr = (lane >> 2) + h2 * 16, ch = (lane & 3u) * 8;
        const uint32_t row = row0 + mt * 32 + rr;
        u32x4_t t = *reinterpret_cast<const u32x4_t*>(patch + rr * kPatchRow + ch);
        if (residual) {
          const u32x4_t rv = rres[mt][o][h2];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            t[e] = pack_bf16x2(bf16_lo(t[e]) + bf16_lo(rv[e]), bf16_hi(t[e]) + bf16_hi(rv[e]));
        }
        if (row < M) *reinterpret_cast<u32x4_t*>(y_wg + ((row - wg_row0) * ldy + col0 + (cg * OTW + o) * 32 + ch)) = t;
      }
    }
}

template <int N, int MT>
static int launch_ys(const uint16_t* x, uint32_t ldx, const uint16_t* w, const uint16_t* bias, const uint16_t* residual,
                     uint32_t ldr, uint16_t* y, uint32_t ldy, uint32_t M, uint32_t NT, uint32_t K, int device,
                     hipStream_t s) {
  constexpr size_t lds = YsGeom<N, MT>::lds_bytes();
  static_assert(lds <= 160 * 1024, "chunk buffers exceed the LDS of a compute unit");
  static bool attr_set[64] = {};
  auto kern = ystat_linear_kernel<N, MT>;
  if (device < 0 || device >= 64 || !attr_set[device]) {
    F3D_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (device >= 0 && device < 64) attr_set[device] = true;
  }
  hipLaunchKernelGGL(kern, dim3(cdiv_u32(M, 128 * MT) * (NT / N)), dim3(64 * kYsWaves), lds, s, x, ldx, w, bias, residual, ldr,
                     y, ldy, M, K, NT);
  return F3D_OK;
}

// Returns F3D_OK when launched, F3D_ERR_UNSUPPORTED when the shape is not covered (the caller then uses the tiled
// GEMM), another code on failure.  Covered: no activation, N a multiple of 128, K a multiple of 64 from 192 up, a bias
// that can be read in 8-byte pieces (the entry point asks that of no bias), row offsets inside a workgroup's panel that fit
// 32 bits.
int launch_ystat_linear(const uint16_t* x, uint32_t ldx, const uint16_t* w, const uint16_t* bias,
                        const uint16_t* residual, uint32_t ldr, uint16_t* y, uint32_t ldy, uint32_t M, uint32_t N,
                        uint32_t K, uint32_t act, int device, hipStream_t s) {
  if (act != F3D_ACT_NONE || N % 128 != 0 || K < 192 || K % 64 != 0 || ((uintptr_t)bias & 7u) != 0) return F3D_ERR_UNSUPPORTED;
  if ((uint64_t)K * 2 * 8 >= (1ull << 32) || (uint64_t)256 * ldx * 2 >= (1ull << 31) ||
      (uint64_t)256 * std::max(ldy, ldr) >= (1ull << 32) || (uint64_t)cdiv_u32(M, 128) * (N / 128) > 0x7FFFF0ull)
    return F3D_ERR_UNSUPPORTED;
  // One workgroup fits a CU.  A panel of 256 x 256 takes about 4 : 3 : 2.2 times as long as one of 256 x 128 and one of
  // 128 x 128 (K = 2048: 49.5, 37, 27.5 us up to 256 panels); the launch takes the form with the least panel time times rounds
  // of the chip.  N = 512, K = 2048: 30,208 rows 64 / 82 / 98 us, 8,192 rows 50 / 37 / 28; N = 128, K = 1024: 120,832 rows
  // (256 x 128, 128 x 128) 57 / 67 us, 32,768 rows 24 / 19.
  // A y that lies on x is taken only where one workgroup holds all columns of its rows, and so reads them before it stores.
  const uint32_t rows2 = cdiv_u32(M, 256), rows1 = cdiv_u32(M, 128);
  const bool in_place = rows_overlap(x, ldx, K, y, ldy, N, M);
  if (in_place && N > 256) return F3D_ERR_UNSUPPORTED;
  auto cost = [](uint64_t panels, uint32_t weight) { return (panels + 255) / 256 * weight; };
  const uint64_t wide = N % 256 == 0 ? cost((uint64_t)rows2 * (N / 256), 20) : ~0ull;
  const uint64_t tall = cost((uint64_t)rows2 * (N / 128), 15), small = cost((uint64_t)rows1 * (N / 128), 11);
  // Up to half as many 128 x 128 panels as an MI355X has CUs (256): 128 x 64 ones, three quarters of the bytes a chunk and twice the CUs that
  // ask for them.  K = 2048, N = 512, in us: 1,536 rows 22.0 -> 19.5, 4,096 rows 23.3 -> 20.6, but 8,192 rows 29 -> 39 (two
  // rounds); K = 1024, N = 256: 5,632 rows 12.7 -> 11.4.
  if (!in_place && 2u * (uint64_t)rows1 * (N / 128) <= 256)
    return launch_ys<64, 1>(x, ldx, w, bias, residual, ldr, y, ldy, M, N, K, device, s);
  if ((in_place && N == 256) || (wide <= tall && wide <= small)) return launch_ys<256, 2>(x, ldx, w, bias, residual, ldr, y, ldy, M, N, K, device, s);
  if (tall <= small) return launch_ys<128, 2>(x, ldx, w, bias, residual, ldr, y, ldy, M, N, K, device, s);
  return launch_ys<128, 1>(x, ldx, w, bias, residual, ldr, y, ldy, M, N, K, device, s);
}

}  // namespace f3d
