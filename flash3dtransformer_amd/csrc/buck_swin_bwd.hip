// Bucketed (scoped) multi-head attention backward for gfx950: any scope size, head_dim 16 / 32 / 64 / 128, optional
// per-bucket valid lengths.
//
// Counterpart of pshattn.buck_swin_bwd (declared src/f3d_frontend.cu:94-97, called from flash3dxfmr/layers/buck_swin.py:69-95;
// the reference ships no kernel source for it, its tests differentiate an SDPA oracle, tests/test_attn_bwd.py: B,L,H,D =
// 4,8192,4,{64,128} with one scope over all buckets, and its model runs buckets of 512 in scopes of 8,
// tests/test_psh_hourglass.py:56-57).  Per batch row, scope and head, with P = softmax(Q Kt / sqrt(D)) recomputed from the
// saved LSE:
//   Delta = rowsum(dO * O)   dV = Pt dO   dP = dO Vt   dS = P * (dP - Delta)   dQ = dS K / sqrt(D)   dK = dSt Q / sqrt(D)
//
// Two kernels, no atomics (every output row is written by exactly one wave):
//   dq    : a workgroup of 4 waves owns 128 QUERIES of one (batch, scope, head) (Q, dO rows in registers, LSE and Delta one
//           scalar per lane) and walks the scope's key tiles (K and V rows through LDS); St = K Qt, dPt = V dOt,
//           dQt += Kt dSt with Kt read transposed.  It runs first and forms Delta on the way.
//   dkdv  : a wave owns 32 or 64 KEYS (K and V rows in registers as MFMA B operands) and walks the scope's query tiles
//           (Q and dO rows, LSE and Delta through LDS).  S = Q Kt and dP = dO Vt come out with a lane holding one key and
//           16 queries, so P and dS (bf16) already are the B operands of dVt += dOt P and dKt += Qt dS, whose A
//           operands (dOt, Qt) are read transposed from LDS (ds_read_b64_tr_b16).
// LDS rows are unpadded with their 16-byte pieces XOR-swizzled (conflict-free 128-bit operand reads); the transposing
// reads address 8-byte pieces per lane and apply the same swizzle to their addresses.
// Valid lengths (kv_len, may be null): keys at in-bucket position >= kv_len[bucket] have P = 0, and so have query rows
// there (the forward gave them O = 0, LSE = 0): their gradients are zero and they add nothing to dK / dV.  Masked rows of
// q, k, v, o, dO and LSE may hold anything: the tiles repeat the last valid row instead of reading them.
//
// What bounds it: mostly vector issue.  A 32 x 32 block at D = 32 (32 exponentials, 16 conversions, 112 multiply-type
// instructions and 14 matrix products over the two kernels) keeps a SIMD's vector ALU active for 880 clocks and takes 1,120
// in scopes of 4,096 rows (counters: dK / dV 73 % of 615 clocks, dQ 86 % of 503); in scopes of 512 it is 970 of 1,560, where
// loading the wave's own rows and storing its gradients weigh against 16 blocks instead of 128.
// Hence: masking costs nothing in the loops (an infinite LSE for masked queries, 8 ANDs in a bucket's
// last key tile; a masked key or query of the wave itself spoils only its own column and is zeroed by the store), the walk
// over buckets has no division, the LSE is brought to the exponent's units once per tile by the wave that loaded it, up to
// four 32-row sub-tiles share a barrier, and all streamed data including LSE and Delta arrives by direct loads (passing LSE
// and Delta through registers made one wave wait for memory in every tile).
// Delta is subtracted behind the dP product.  As the product's start value it would save 32 subtractions a block (122,880
// rows in scopes of 4,096: 275 us instead of 292), but dP - Delta then rounds differently, and the backward of batch
// statistics enlarges the flipped last bits of dS to 1e-3 of a model's gradients.
// The sub-tile loop stays rolled: unrolled, the accumulators cost up to 128 registers more and half the occupancy.
// Keeping a whole scope in LDS (one 16-wave workgroup per scope) is slower at 256 / 512 tokens too, and so were separate
// Delta, dK / dV and dQ kernels.  Measured, both kernels, against those: 8 heads x 131,072 rows, 512-row scopes 430 -> 382 us,
// with valid lengths of 3/4 to full buckets 538 -> 342; scopes of 8 x 512, 122,880 rows 524 -> 292, 24,576 rows 263 -> 126;
// 20,480 rows of 512-row scopes 39 -> 24; 4 heads of 64, 65,536 rows: 236 -> 154, of 128, 32,768 rows: 257 -> 208.
// The score products of both key tiles of a wave are issued before the first exponential, and gradients leave in 16-byte
// pieces (the halves of a wave exchange registers; 8-byte pieces touched twice the lines per store): 482,304 rows of 512-row scopes
// 182 -> 175 us, 30,208 rows x 16 heads 181 -> 171, 8 heads x 131,072 rows 405 -> 390, in 256-row scopes 269 -> 253, 64-wide
// heads 158 -> 148, same bits.  One kernel for dQ, dK and dV (five products a block instead of seven, dQ summed in LDS by eight waves
// that pass its tiles on) reached 340 at 8 heads x 131,072 rows, but 35 instead of 25 at 20,480 rows: with both P and dS turned
// round through LDS, two waves a SIMD and a hand-over per tile, a step took 3,400 clocks for 2,000 of vector issue.
#include <algorithm>
#include "f3d_device.h"
#include "f3d_internal.h"

namespace f3d {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

constexpr int kStreamWaves = 4;
constexpr int kStreamXcd = 8;
constexpr int kStreamCus = 256;

template <int D>
struct SGeom {
  static constexpr int KSTEPS = D / 16;
  static constexpr int DT = D < 32 ? 1 : D / 32;   // 32-feature output tiles
  static constexpr int CPK = D / 8;                // 16-byte pieces per row
  static constexpr int ROWB = D * 2;               // bytes per row
  static constexpr int RPB = 1024 / ROWB;          // rows one direct-load instruction fills
  static constexpr int NSUB = D <= 32 ? 4 : D <= 64 ? 2 : 1;   // 32-row sub-tiles streamed per barrier
  static constexpr int SWZ_DIV = 16 / CPK;         // rows sharing one swizzle value
  static constexpr int TILEB = 32 * ROWB;          // bytes of a 32-row tile
};

// 16 (4) bytes per lane from global memory straight into LDS: lane l of the wave lands at lds_addr + 16 l (4 l).
__device__ __forceinline__ void stream_dma16(const void* gbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(gbase)
               : "memory", "m0");
}
__device__ __forceinline__ void stream_dma4(const void* gbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(gbase)
               : "memory", "m0");
}

// Two runs of ROWS consecutive rows (g0, ld0 bytes a row; g1, ld1) -> two swizzled LDS tiles, one behind the other; the
// direct loads are shared by the workgroup's waves.  Rows past `last` are copies of row `last`: what lies there in memory
// (masked rows, which may hold anything) is not read.
template <int D, int ROWS>
__device__ __forceinline__ void stream_fill_pair(const char* g0, uint32_t ld0, const char* g1, uint32_t ld1,
                                                 uint32_t last, uint32_t lds_tile, uint32_t wave, uint32_t lane) {
  using G = SGeom<D>;
  constexpr int BLK = ROWS / G::RPB;
  const uint32_t r = lane / G::CPK, pos = lane % G::CPK;
#pragma unroll
  for (int i = 0; i < (2 * BLK + kStreamWaves - 1) / kStreamWaves; ++i) {
    const uint32_t n = wave + i * kStreamWaves;       // uniform
    if (n < 2u * BLK) {
      const bool second = n >= (uint32_t)BLK;
      const uint32_t blk = second ? n - BLK : n, ld = second ? ld1 : ld0;
      const uint32_t ck = pos ^ (((blk * G::RPB + r) / G::SWZ_DIV) & (G::CPK - 1));
      const uint32_t row0 = min(blk * G::RPB, last);
      const uint64_t g = (uint64_t)(uintptr_t)(second ? g1 : g0) + (uint64_t)row0 * ld;
      const uint64_t gu = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)g) |
                          ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(g >> 32)) << 32);
      stream_dma16(reinterpret_cast<const void*>((uintptr_t)gu), min(r, last - row0) * ld + ck * 16u,
                   __builtin_amdgcn_readfirstlane(lds_tile + n * 1024u));
    }
  }
}

// the lane's byte offset of its 8-byte piece for the transposing reads of feature tile dt: row 4 half + l16 / 4 +
// 8 hi of a 32-row tile, features 32 dt + d_base + 4 (l16 % 4) .. + 3, the row's swizzle applied to the piece index
template <int D>
__device__ __forceinline__ uint32_t stream_tr_offset(uint32_t lane, uint32_t hi, uint32_t dt) {
  using G = SGeom<D>;
  const uint32_t half = lane >> 5, l16 = lane & 15u, d_base = 16u * ((lane >> 4) & 1u);
  const uint32_t row = 4u * half + l16 / 4u + 8u * hi;
  const uint32_t colb = (32u * dt + d_base + 4u * (l16 & 3u)) * 2u;         // byte column, a multiple of 8
  const uint32_t piece = (colb / 16u) ^ ((row / G::SWZ_DIV) & (G::CPK - 1));
  return row * G::ROWB + piece * 16u + (colb & 8u);
}

// A operand read transposed from a swizzled LDS tile of 32 rows: lane (m = feature of tile dt) gets, for k-step kk,
// slots 0..3 = rows 16 kk + 4 half + 0..3 and slots 4..7 = the same + 8 (the order in which an accumulator tile hands
// its rows to the next MFMA as a B operand).  Adding 16 rows leaves a row's swizzle value unchanged.
template <int D>
__device__ __forceinline__ void stream_load_tr(const char* tile, uint32_t tr_lo, uint32_t tr_hi, bool tr_lane,
                                               bf16x8_t (&f)[2]) {
  constexpr int ROWB = SGeom<D>::ROWB;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    i16x4_t lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
    if (tr_lane) {
      lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(tile + tr_lo + (kk * 16) * ROWB));
      hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(tile + tr_hi + (kk * 16) * ROWB));
    }
    f[kk] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}

struct StreamItem {
  uint32_t batch, scope, head, blk;
};
// Workgroups go round the XCDs in launch order: consecutive work units (the blocks of an item read the same streamed
// rows) are given to one XCD, so that its L2 serves them.  false: past the end.
__device__ __forceinline__ bool stream_item(uint32_t num_scope, uint32_t num_head, uint32_t n_blk, uint32_t n_unit,
                                            StreamItem& it) {
  const uint32_t per_xcd = gridDim.x / kStreamXcd;
  const uint32_t unit = blockIdx.x % kStreamXcd * per_xcd + blockIdx.x / kStreamXcd;
  if (unit >= n_unit) return false;
  const uint32_t item = unit / n_blk;
  it.blk = unit - item * n_blk;
  it.head = item % num_head;
  it.scope = (item / num_head) % num_scope;
  it.batch = item / (num_head * num_scope);
  return true;
}

// bucket ids and valid lengths of the scope -> LDS; returns false (uniformly) when an id lies outside the sequence:
// such a scope contributes nothing, as in the forward's backward-facing contract
__device__ __forceinline__ bool stream_scope_table(const uint32_t* scope_buckets, const int32_t* kv_len, uint32_t scope,
                                                   uint32_t scope_size, uint32_t bs, uint32_t n_bucket,
                                                   uint32_t* s_bucket, int32_t* s_len) {
  int bad = 0;
  for (uint32_t j = threadIdx.x; j < scope_size; j += blockDim.x) {
    const uint32_t b = scope_buckets[(size_t)scope * scope_size + j];
    s_bucket[j] = b;
    if (b >= n_bucket) bad = 1;
    s_len[j] = b >= n_bucket ? 0 : (kv_len ? min(max(kv_len[b], 0), (int32_t)bs) : (int32_t)bs);
  }
  return __syncthreads_or(bad) == 0;
}

// Walk over the tiles of ROWS rows of a scope that hold valid rows, bucket by bucket (all members uniform)
template <int ROWS>
struct StreamWalk {
  const uint32_t* s_bucket;
  const int32_t* s_len;
  uint32_t scope_size, bs, j, r, len, row0;   // tile: rows [r, r + ROWS) of bucket j, which starts at row0
  __device__ __forceinline__ StreamWalk(const uint32_t* sb, const int32_t* sl, uint32_t n, uint32_t bucket_size)
      : s_bucket(sb), s_len(sl), scope_size(n), bs(bucket_size), j(0u), r(0u) {
    load();
    if (len == 0) next();
  }
  __device__ __forceinline__ void load() {
    len = __builtin_amdgcn_readfirstlane((uint32_t)s_len[j]);
    row0 = __builtin_amdgcn_readfirstlane(s_bucket[j]) * bs;
  }
  __device__ __forceinline__ bool done() const { return j >= scope_size; }
  __device__ __forceinline__ void next() {
    r += ROWS;
    while (r >= len) {
      r = 0;
      if (++j >= scope_size) return;
      load();
    }
  }
};

// LDS: two buffers of two tiles of 32 NSUB rows, then per buffer 32 NSUB LSE and Delta (dkdv), then the scope table
template <int D>
constexpr size_t stream_lds_bytes(uint32_t scope_size) {
  return (size_t)4 * SGeom<D>::TILEB * SGeom<D>::NSUB + (size_t)4 * 32 * SGeom<D>::NSUB * 4 + (size_t)scope_size * 8;
}

// a 32 x 32 accumulator tile (transposed output: the lane's row, features 8 g + 4 half .. + 3 per group g) as bf16 in 16-byte pieces:
// the lower half-wave's second group is exchanged with the upper half-wave's first, so that a lane holds 8 consecutive features
template <int N>
__device__ __forceinline__ void store_features(uint16_t* row, uint32_t half, const f32x16_t& x, float f, bool ok) {
#pragma unroll
  for (int g = 0; g < N / 8; g += 2) {
    uint32_t w[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 2; ++e) w[h][e] = ok ? pack_bf16x2(x[(g + h) * 4 + 2 * e] * f, x[(g + h) * 4 + 2 * e + 1] * f) : 0u;
    const auto lo = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
    *reinterpret_cast<u32x4_t*>(row + (g + half) * 8) = u32x4_t{lo[0], hi[0], lo[1], hi[1]};
  }
}

// ---- Delta, dQ ------------------------------------------------------------------------------------------------
// Runs first: Delta of the wave's queries is formed from its O and dO rows (dO is in registers anyway).
template <int D>
__global__ __launch_bounds__(64 * kStreamWaves, D > 64 ? 1 : D > 32 ? 2 : 4) void bwd_dq_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, uint32_t ld,
    const uint16_t* __restrict__ o, const uint16_t* __restrict__ d_o, const float* __restrict__ lse,
    float* __restrict__ delta, uint16_t* __restrict__ dq, const uint32_t* __restrict__ scope_buckets, uint32_t num_scope,
    uint32_t scope_size, uint32_t bs, uint32_t seq_len, uint32_t num_head, const int32_t* __restrict__ kv_len,
    float scale, float scale_log2, uint32_t ldg, uint32_t n_blk, uint32_t n_unit) {
  using G = SGeom<D>;
  constexpr int KSTEPS = G::KSTEPS, ROWB = G::ROWB, DT = G::DT, NSUB = G::NSUB, ROWS = 32 * NSUB, TILEB = G::TILEB * NSUB;
  extern __shared__ __attribute__((aligned(16))) char lds_s[];
  uint32_t* s_bucket = reinterpret_cast<uint32_t*>(lds_s + 4 * TILEB + 4 * ROWS * 4);
  int32_t* s_len = reinterpret_cast<int32_t*>(s_bucket + scope_size);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds_s;

  StreamItem it;
  if (!stream_item(num_scope, num_head, n_blk, n_unit, it)) return;
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t lq = lane & 31u, half = lane >> 5;
  const uint32_t n_bucket = seq_len / bs;
  const bool good = stream_scope_table(scope_buckets, kv_len, it.scope, scope_size, bs, n_bucket, s_bucket, s_len);

  const uint32_t ldo = num_head * D;
  const size_t base_qkv = (size_t)it.batch * seq_len * ld + (size_t)it.head * D;
  const size_t base_o = (size_t)it.batch * seq_len * ldo + (size_t)it.head * D;
  const size_t base_l = (size_t)it.batch * seq_len * num_head + it.head;

  // this wave's 32 queries, all of one bucket
  const uint32_t qloc0 = (it.blk * kStreamWaves + wave) * 32u;
  const uint32_t qj = qloc0 / bs, q_in_b0 = qloc0 - qj * bs;
  const uint32_t q_bucket = __builtin_amdgcn_readfirstlane(s_bucket[qj]);
  const uint32_t qrow = q_bucket * bs + q_in_b0 + lq;
  const int32_t q_len = __builtin_amdgcn_readfirstlane(s_len[qj]) - (int32_t)q_in_b0;   // valid ones of the wave's queries
  bf16x8_t qf[KSTEPS], dof[KSTEPS];
  float lse2, dlt;
  if (q_bucket < n_bucket) {
    const uint16_t* qr = q + base_qkv + (size_t)qrow * ld + half * 8;
    const uint16_t* dr = d_o + base_o + (size_t)qrow * ldo + half * 8;
    const uint16_t* orow = o + base_o + (size_t)qrow * ldo + half * 8;
    dlt = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      qf[ks] = *reinterpret_cast<const bf16x8_t*>(qr + ks * 16);
      dof[ks] = *reinterpret_cast<const bf16x8_t*>(dr + ks * 16);
      const u32x4_t ov = *reinterpret_cast<const u32x4_t*>(orow + ks * 16);
      const u32x4_t dv = __builtin_bit_cast(u32x4_t, dof[ks]);
      // one sum over the row's features in ascending order: 8 of them in the lane with half 0, the next 8 in the other
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        float sum = dlt;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sum = __builtin_fmaf(bf16_lo(ov[e]), bf16_lo(dv[e]), sum);
          sum = __builtin_fmaf(bf16_hi(ov[e]), bf16_hi(dv[e]), sum);
        }
        dlt = __shfl(sum, lq + 32u * h);
      }
    }
    lse2 = lse[base_l + (size_t)qrow * num_head] * 1.4426950408889634f;
    if (half == 0) delta[base_l + (size_t)qrow * num_head] = dlt;
  }
  if (!good) return;

  const uint32_t dir_off = lq * ROWB + ((half ^ ((lq / G::SWZ_DIV) & (G::CPK - 1))) * 16u);   // k-step ks: ^ (ks * 32)
  uint32_t tr_lo[DT], tr_hi[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    tr_lo[dt] = stream_tr_offset<D>(lane, 0, dt);
    tr_hi[dt] = stream_tr_offset<D>(lane, 1, dt);
  }
  const bool tr_lane = D >= 32 || 16u * ((lane >> 4) & 1u) < (uint32_t)D;

  f32x16_t acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  // one 32-key sub-tile; keys at or past k_valid get dS = 0 (a query's lane holds nothing of another query: those past
  // the valid length are left to the store)
  auto step = [&](const char* sK, const char* sV, int32_t k_valid) {
    bf16x8_t ka[KSTEPS], va[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      ka[ks] = *reinterpret_cast<const bf16x8_t*>(sK + (dir_off ^ (ks * 32u)));
      va[ks] = *reinterpret_cast<const bf16x8_t*>(sV + (dir_off ^ (ks * 32u)));
    }
    // register i of a lane is key (i/4)*8 + 4 half + i%4 of the tile, for the lane's query
    uint32_t sb[8];
    f32x16_t s_acc, p_acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) { s_acc[i] = 0.f; p_acc[i] = 0.f; }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[ks], qf[ks], s_acc, 0, 0, 0);    // St[key][query]
      p_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[ks], dof[ks], p_acc, 0, 0, 0);   // dPt[key][query]
    }
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      float ds[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        ds[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[i + e], scale_log2, -lse2)) * (p_acc[i + e] - dlt);
      sb[i / 2] = pack_bf16x2(ds[0], ds[1]);
    }
    if (k_valid < 32) {      // uniform, a bucket's last tile
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int32_t left = k_valid - (int32_t)((i / 2) * 8 + half * 4 + (i % 2) * 2);   // of the pair's two keys
        const uint32_t keep = left >= 2 ? 0xFFFFFFFFu : left == 1 ? 0x0000FFFFu : 0u;
        sb[i] &= keep;
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      bf16x8_t ktr[2];
      stream_load_tr<D>(sK, tr_lo[dt], tr_hi[dt], tr_lane, ktr);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const u32x4_t sraw = {sb[kk * 4 + 0], sb[kk * 4 + 1], sb[kk * 4 + 2], sb[kk * 4 + 3]};
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktr[kk], __builtin_bit_cast(bf16x8_t, sraw), acc[dt], 0, 0, 0);
      }
    }
  };

  StreamWalk<ROWS> w(s_bucket, s_len, scope_size, bs);
  auto fill = [&](uint32_t b) {   // the walk's tile -> buffer b
    const size_t grow = w.row0 + w.r;
    const uint32_t last = min(w.len - w.r, (uint32_t)ROWS) - 1u;
    stream_fill_pair<D, ROWS>(reinterpret_cast<const char*>(k + base_qkv + grow * ld), ld * 2u,
                              reinterpret_cast<const char*>(v + base_qkv + grow * ld), ld * 2u, last, lds0 + b * 2u * TILEB, wave, lane);
  };
  uint32_t b = 0;
  if (!w.done()) fill(b);
  while (!w.done()) {
    const int32_t k_valid = (int32_t)(w.len - w.r);
    __builtin_amdgcn_s_waitcnt(0);   // this wave's loads of the tile have landed
    __syncthreads();                 // ... everybody's; and everybody has left the other buffer
    w.next();
    if (!w.done()) fill(b ^ 1u);
    const char* sK = lds_s + b * 2u * TILEB;
    if (q_len > 0) {
#pragma unroll 1
      for (int u = 0; u < NSUB && k_valid > 32 * u; ++u)
        step(sK + u * G::TILEB, sK + TILEB + u * G::TILEB, k_valid - 32 * u);
    }
    b ^= 1u;
  }
  const size_t base_g = (size_t)it.batch * seq_len * ldg + (size_t)it.head * D;
  uint16_t* dqrow = dq + base_g + (size_t)qrow * ldg;
  const bool q_ok = (int32_t)lq < q_len;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) store_features<D < 32 ? D : 32>(dqrow + dt * 32, half, acc[dt], scale, q_ok);
}

// ---- dK, dV -------------------------------------------------------------------------------------------------
template <int D, int KT>
__global__ __launch_bounds__(64 * kStreamWaves, D > 64 ? 1 : D > 32 || KT > 1 ? 2 : D > 16 ? 4 : 3) void bwd_dkdv_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, uint32_t ld,
    const uint16_t* __restrict__ d_o, const float* __restrict__ lse, const float* __restrict__ delta,
    uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, const uint32_t* __restrict__ scope_buckets,
    uint32_t num_scope, uint32_t scope_size, uint32_t bs, uint32_t seq_len, uint32_t num_head,
    const int32_t* __restrict__ kv_len, float scale, float scale_log2, uint32_t ldg, uint32_t n_blk, uint32_t n_unit) {
  using G = SGeom<D>;
  constexpr int KSTEPS = G::KSTEPS, ROWB = G::ROWB, DT = G::DT, NSUB = G::NSUB, ROWS = 32 * NSUB, TILEB = G::TILEB * NSUB;
  extern __shared__ __attribute__((aligned(16))) char lds_s[];
  float* s_lse = reinterpret_cast<float*>(lds_s + 4 * TILEB);
  float* s_delta = s_lse + 2 * ROWS;
  uint32_t* s_bucket = reinterpret_cast<uint32_t*>(s_delta + 2 * ROWS);
  int32_t* s_len = reinterpret_cast<int32_t*>(s_bucket + scope_size);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds_s;

  StreamItem it;
  if (!stream_item(num_scope, num_head, n_blk, n_unit, it)) return;
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t lq = lane & 31u, half = lane >> 5;
  const uint32_t n_bucket = seq_len / bs;
  if (!stream_scope_table(scope_buckets, kv_len, it.scope, scope_size, bs, n_bucket, s_bucket, s_len)) return;

  const uint32_t ldo = num_head * D;   // dO is dense [B, L, H, D]
  const size_t base_qkv = (size_t)it.batch * seq_len * ld + (size_t)it.head * D;
  const size_t base_o = (size_t)it.batch * seq_len * ldo + (size_t)it.head * D;
  const size_t base_l = (size_t)it.batch * seq_len * num_head + it.head;

  // this wave's 32 KT keys, all of one bucket; lane -> keys lq, lq + 32, ..
  const uint32_t kloc0 = (it.blk * kStreamWaves + wave) * 32u * KT;
  const uint32_t kj = kloc0 / bs, k_in_b0 = kloc0 - kj * bs;
  const uint32_t krow = __builtin_amdgcn_readfirstlane(s_bucket[kj]) * bs + k_in_b0 + lq;   // row inside the sequence
  const int32_t k_len = __builtin_amdgcn_readfirstlane(s_len[kj]) - (int32_t)k_in_b0;       // valid ones of the wave's keys
  bf16x8_t kf[KT][KSTEPS], vf[KT][KSTEPS];
#pragma unroll
  for (int a = 0; a < KT; ++a) {
    const uint16_t* kr = k + base_qkv + (size_t)(krow + 32u * a) * ld + half * 8;
    const uint16_t* vr = v + base_qkv + (size_t)(krow + 32u * a) * ld + half * 8;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      kf[a][ks] = *reinterpret_cast<const bf16x8_t*>(kr + ks * 16);
      vf[a][ks] = *reinterpret_cast<const bf16x8_t*>(vr + ks * 16);
    }
  }

  const uint32_t dir_off = lq * ROWB + ((half ^ ((lq / G::SWZ_DIV) & (G::CPK - 1))) * 16u);   // k-step ks: ^ (ks * 32)
  uint32_t tr_lo[DT], tr_hi[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    tr_lo[dt] = stream_tr_offset<D>(lane, 0, dt);
    tr_hi[dt] = stream_tr_offset<D>(lane, 1, dt);
  }
  const bool tr_lane = D >= 32 || 16u * ((lane >> 4) & 1u) < (uint32_t)D;

  f32x16_t acc_dk[KT][DT], acc_dv[KT][DT];
#pragma unroll
  for (int a = 0; a < KT; ++a)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) { acc_dk[a][dt][i] = 0.f; acc_dv[a][dt][i] = 0.f; }

  // one 32-query sub-tile (a key's lane holds nothing of another key: those past the valid length are left to the store)
  auto step = [&](const char* sQ, const char* sD, const float* lse_t, const float* dlt_t) {
    bf16x8_t qa[KSTEPS], da[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      qa[ks] = *reinterpret_cast<const bf16x8_t*>(sQ + (dir_off ^ (ks * 32u)));
      da[ks] = *reinterpret_cast<const bf16x8_t*>(sD + (dir_off ^ (ks * 32u)));
    }
    // register i of a lane is query (i/4)*8 + 4 half + i%4 of the tile, for the lane's key
    float lse2[16], dl[16];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const float4 l4 = *reinterpret_cast<const float4*>(lse_t + g4 * 8 + half * 4);
      const float4 d4 = *reinterpret_cast<const float4*>(dlt_t + g4 * 8 + half * 4);
      const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dv4[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) { lse2[g4 * 4 + r] = lv[r]; dl[g4 * 4 + r] = dv4[r]; }
    }
    uint32_t pb[KT][8], sb[KT][8];
    f32x16_t s_all[KT], p_all[KT];
#pragma unroll
    for (int a = 0; a < KT; ++a) {
#pragma unroll
      for (int i = 0; i < 16; ++i) { s_all[a][i] = 0.f; p_all[a][i] = 0.f; }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        s_all[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[ks], kf[a][ks], s_all[a], 0, 0, 0);   // S[query][key]
        p_all[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(da[ks], vf[a][ks], p_all[a], 0, 0, 0);   // dP[query][key]
      }
    }
    if constexpr (KT > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < KT; ++a) {
      const f32x16_t &s_acc = s_all[a], &p_acc = p_all[a];
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        float p[2], ds[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[i + e], scale_log2, -lse2[i + e]));
          ds[e] = p[e] * (p_acc[i + e] - dl[i + e]);
        }
        pb[a][i / 2] = pack_bf16x2(p[0], p[1]);
        sb[a][i / 2] = pack_bf16x2(ds[0], ds[1]);
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      bf16x8_t dot[2], qtr[2];
      stream_load_tr<D>(sD, tr_lo[dt], tr_hi[dt], tr_lane, dot);
      stream_load_tr<D>(sQ, tr_lo[dt], tr_hi[dt], tr_lane, qtr);
#pragma unroll
      for (int a = 0; a < KT; ++a)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const u32x4_t praw = {pb[a][kk * 4 + 0], pb[a][kk * 4 + 1], pb[a][kk * 4 + 2], pb[a][kk * 4 + 3]};
          const u32x4_t sraw = {sb[a][kk * 4 + 0], sb[a][kk * 4 + 1], sb[a][kk * 4 + 2], sb[a][kk * 4 + 3]};
          acc_dv[a][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dot[kk], __builtin_bit_cast(bf16x8_t, praw), acc_dv[a][dt], 0, 0, 0);
          acc_dk[a][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qtr[kk], __builtin_bit_cast(bf16x8_t, sraw), acc_dk[a][dt], 0, 0, 0);
        }
    }
  };

  StreamWalk<ROWS> w(s_bucket, s_len, scope_size, bs);
  auto fill = [&](uint32_t b) {   // the walk's tile -> buffer b
    const size_t grow = w.row0 + w.r;
    const uint32_t last = min(w.len - w.r, (uint32_t)ROWS) - 1u;
    stream_fill_pair<D, ROWS>(reinterpret_cast<const char*>(q + base_qkv + grow * ld), ld * 2u,
                              reinterpret_cast<const char*>(d_o + base_o + grow * ldo), ldo * 2u, last, lds0 + b * 2u * TILEB, wave, lane);
    // LSE and Delta of the tile's rows by direct loads too: through registers one wave would wait for memory in every tile
    constexpr uint32_t LROWS = ROWS < 64 ? ROWS : 64;      // rows of one direct load
    const uint32_t arr = wave & 1u, part = wave >> 1;
    if (part * LROWS < (uint32_t)ROWS && lane < LROWS) {
      const uint32_t part0 = min(part * LROWS, last);
      const uint64_t g = (uint64_t)(uintptr_t)((arr ? delta : lse) + base_l + (grow + part0) * num_head);
      const uint64_t gu = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)g) |
                          ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(g >> 32)) << 32);
      stream_dma4(reinterpret_cast<const void*>((uintptr_t)gu), min(lane, last - part0) * num_head * 4u,
                  __builtin_amdgcn_readfirstlane(lds0 + 4u * TILEB + ((arr * 2u + b) * ROWS + part * LROWS) * 4u));
    }
  };
  uint32_t b = 0;
  if (!w.done()) fill(b);
  while (!w.done()) {
    const int32_t q_valid = (int32_t)(w.len - w.r);
    __builtin_amdgcn_s_waitcnt(0);   // this wave's loads of the tile have landed
    // the LSE in the exponent's units, by the wave that loaded it (waves 0 and 2); queries past the bucket's valid length get
    // an infinite one, which makes their P and dS zero
    if ((wave & 1u) == 0u) {
      const uint32_t i = (wave >> 1) * 64u + lane;
      if (i < (uint32_t)ROWS) {
        const float l = s_lse[b * ROWS + i] * 1.4426950408889634f;
        s_lse[b * ROWS + i] = (int32_t)i < q_valid ? l : __builtin_inff();
      }
    }
    __syncthreads();                 // ... everybody's; and everybody has left the other buffer
    w.next();
    if (!w.done()) fill(b ^ 1u);
    const char* sQ = lds_s + b * 2u * TILEB;
    const float *lse_t = s_lse + b * ROWS, *dlt_t = s_delta + b * ROWS;
    if (k_len > 0) {
#pragma unroll 1
      for (int u = 0; u < NSUB && q_valid > 32 * u; ++u)
        step(sQ + u * G::TILEB, sQ + TILEB + u * G::TILEB, lse_t + 32 * u, dlt_t + 32 * u);
    }
    b ^= 1u;
  }

  // acc[a][dt][g4*4 + r] = d?t[feature 32 dt + g4*8 + 4 half + r][key 32 a + lq]: 4 consecutive features of a key per group
  // the gradients' rows are ldg elements apart (dense: ldg = ldo; thirds of one [B, L, 3 H D] tensor: ldg = 3 ldo)
  const size_t base_g = (size_t)it.batch * seq_len * ldg + (size_t)it.head * D;
#pragma unroll
  for (int a = 0; a < KT; ++a) {
    uint16_t* dkrow = dk + base_g + (size_t)(krow + 32u * a) * ldg;
    uint16_t* dvrow = dv + base_g + (size_t)(krow + 32u * a) * ldg;
    const bool key_ok = (int32_t)(32u * a + lq) < k_len;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      store_features<D < 32 ? D : 32>(dkrow + dt * 32, half, acc_dk[a][dt], scale, key_ok);
      store_features<D < 32 ? D : 32>(dvrow + dt * 32, half, acc_dv[a][dt], 1.0f, key_ok);
    }
  }
}

template <int D, int KT>
static int launch_stream(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint32_t ld, const uint16_t* o,
                         const uint16_t* d_o, const float* lse, float* delta, uint16_t* dq, uint16_t* dk, uint16_t* dv,
                         const uint32_t* scope_buckets, uint32_t num_scope, uint32_t scope_size, uint32_t bs,
                         uint32_t batch, uint32_t seq_len, uint32_t num_head, const int32_t* kv_len, uint32_t ldg,
                         hipStream_t s) {
  const size_t lds = stream_lds_bytes<D>(scope_size);
  if (lds > 64 * 1024) {
    // the scope table is the only part that grows: 8 bytes per bucket of the scope
    F3D_CHECK_HIP(hipFuncSetAttribute((const void*)bwd_dkdv_kernel<D, KT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    F3D_CHECK_HIP(hipFuncSetAttribute((const void*)bwd_dq_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  }
  const uint32_t scope_tokens = scope_size * bs;
  const uint32_t items = batch * num_scope * num_head;
  const float scale = 1.0f / sqrtf((float)D), scale_log2 = 1.4426950408889634f * scale;
  const dim3 block(64 * kStreamWaves);
  auto grid = [](uint32_t units) { return dim3((units + kStreamXcd - 1) / kStreamXcd * kStreamXcd); };
  const uint32_t q_blk = scope_tokens / (32u * kStreamWaves), k_blk = scope_tokens / (32u * kStreamWaves * KT);
  hipLaunchKernelGGL(bwd_dq_kernel<D>, grid(items * q_blk), block, lds, s, q, k, v, ld, o, d_o, lse, delta, dq,
                     scope_buckets, num_scope, scope_size, bs, seq_len, num_head, kv_len, scale, scale_log2, ldg, q_blk,
                     items * q_blk);
  hipLaunchKernelGGL((bwd_dkdv_kernel<D, KT>), grid(items * k_blk), block, lds, s, q, k, v, ld, d_o, lse, delta, dk,
                     dv, scope_buckets, num_scope, scope_size, bs, seq_len, num_head, kv_len, scale, scale_log2, ldg, k_blk,
                     items * k_blk);
  return F3D_OK;
}

// Backward for any scope size (buckets of a multiple of 128 rows), head_dim 16 / 32 / 64 / 128.
static int launch_attn_bwd(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint32_t ld, const uint16_t* o,
                           const uint16_t* d_o, const float* lse, float* delta, uint16_t* dq, uint16_t* dk, uint16_t* dv,
                           const uint32_t* scope_buckets, uint32_t num_scope, uint32_t scope_size, uint32_t bs,
                           uint32_t batch, uint32_t seq_len, uint32_t num_head, uint32_t head_dim, const int32_t* kv_len,
                           uint32_t ldg, hipStream_t s) {
  if ((uint64_t)batch * num_scope * num_head * (scope_size * bs / (32u * kStreamWaves)) > 0xFFFFF0ull) {
    set_error("attention problem too large for one launch (%llu items)", (unsigned long long)batch * num_scope * num_head);
    return F3D_ERR_INVALID;
  }
#define F3D_STREAM(DD, KT)                                                                                              \
  return launch_stream<DD, KT>(q, k, v, ld, o, d_o, lse, delta, dq, dk, dv, scope_buckets, num_scope, scope_size, bs, batch, \
                               seq_len, num_head, kv_len, ldg, s)
  // 64 keys per wave halve the LDS reads per product where that still gives every CU a workgroup (8 heads x 131,072 rows:
  // 390 us for both kernels against 398; 122,880 rows in scopes of 4,096: 324 against 345), 32 below (24,576 rows in
  // scopes of 4,096, 96 workgroups of 64-key waves: 133 us against 152).  Wider heads leave no registers for 64.
  const uint64_t tokens = (uint64_t)scope_size * bs;
  const bool wide = tokens % 256u == 0 && (uint64_t)batch * num_scope * num_head * (tokens / 256u) >= (uint64_t)kStreamCus;
  switch (head_dim) {
    case 16: if (wide) F3D_STREAM(16, 2); F3D_STREAM(16, 1);
    case 32: if (wide) F3D_STREAM(32, 2); F3D_STREAM(32, 1);
    case 64: F3D_STREAM(64, 1);
    case 128: F3D_STREAM(128, 1);
    default:
      set_error("No backward kernel found for head_dim=%u (supported: 16, 32, 64, 128)", head_dim);
      return F3D_ERR_UNSUPPORTED;
  }
#undef F3D_STREAM
}

}  // namespace f3d
extern "C" int f3d_buck_swin_bwd(const f3d_bf16_t* q, const f3d_bf16_t* k, const f3d_bf16_t* v,
                                 uint32_t qkv_row_stride, const f3d_bf16_t* o, const f3d_bf16_t* d_o,
                                 const float* lse, float* delta, f3d_bf16_t* dq, f3d_bf16_t* dk, f3d_bf16_t* dv,
                                 const uint32_t* scope_buckets, uint32_t num_scope, uint32_t scope_size,
                                 uint32_t bucket_size, uint32_t batch, uint32_t seq_len, uint32_t num_head,
                                 uint32_t head_dim, const int32_t* kv_len, int device, void* stream) {
  return f3d_buck_swin_bwd_strided(q, k, v, qkv_row_stride, o, d_o, lse, delta, dq, dk, dv, num_head * head_dim,
                                   scope_buckets, num_scope, scope_size, bucket_size, batch, seq_len, num_head, head_dim,
                                   kv_len, device, stream);
}

extern "C" int f3d_buck_swin_bwd_strided(const f3d_bf16_t* q, const f3d_bf16_t* k, const f3d_bf16_t* v,
                                         uint32_t qkv_row_stride, const f3d_bf16_t* o, const f3d_bf16_t* d_o,
                                         const float* lse, float* delta, f3d_bf16_t* dq, f3d_bf16_t* dk, f3d_bf16_t* dv,
                                         uint32_t grad_row_stride, const uint32_t* scope_buckets, uint32_t num_scope,
                                         uint32_t scope_size, uint32_t bucket_size, uint32_t batch, uint32_t seq_len,
                                         uint32_t num_head, uint32_t head_dim, const int32_t* kv_len, int device,
                                         void* stream) {
  using namespace f3d;
  F3D_CHECK_ARG(q && k && v && o && d_o && lse && delta && dq && dk && dv && scope_buckets, "null tensor pointer");
  F3D_CHECK_ARG(grad_row_stride >= num_head * head_dim && grad_row_stride % 8 == 0,
                "dq/dk/dv row stride %u must be a multiple of 8 and at least num_head*head_dim=%u", grad_row_stride,
                num_head * head_dim);
  F3D_CHECK_ARG(bucket_size >= 128 && bucket_size % 128 == 0, "bucket_size=%u must be a multiple of 128",
                bucket_size);
  F3D_CHECK_ARG(seq_len % bucket_size == 0, "sequence length %u is not a multiple of bucket_size=%u", seq_len,
                bucket_size);
  F3D_CHECK_ARG(qkv_row_stride >= num_head * head_dim && qkv_row_stride % 8 == 0,
                "q/k/v row stride %u must be a multiple of 8 and at least num_head*head_dim=%u", qkv_row_stride,
                num_head * head_dim);
  F3D_CHECK_ARG((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)d_o | (uintptr_t)dq |
                  (uintptr_t)dk | (uintptr_t)dv) & 15u) == 0,
                "q/k/v/o/dO/dQ/dK/dV must be 16-byte aligned");
  F3D_CHECK_ARG(scope_size >= 1, "scope_size must be at least 1");
  if (!(head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128)) {
    set_error("No backward kernel found for head_dim=%u (supported: 16, 32, 64, 128)", head_dim);
    return F3D_ERR_UNSUPPORTED;
  }
  if ((uint64_t)scope_size * 8 > 32 * 1024) {
    set_error("attention backward: a scope of %u buckets exceeds the 4096 the scope table holds", scope_size);
    return F3D_ERR_UNSUPPORTED;
  }
  if (batch == 0 || num_scope == 0 || num_head == 0) return F3D_OK;
  DeviceGuard guard(device);
  F3D_CHECK_ARG(guard.ok, "cannot select device %d", device);
  hipStream_t s = (hipStream_t)stream;
  SyncBracket sync(s);
  const int rc = launch_attn_bwd(q, k, v, qkv_row_stride, o, d_o, lse, delta, dq, dk, dv, scope_buckets, num_scope, scope_size,
                                 bucket_size, batch, seq_len, num_head, head_dim, kv_len, grad_row_stride, s);
  if (rc != F3D_OK) return rc;
  F3D_CHECK_HIP(hipGetLastError());
  return F3D_OK;
}
