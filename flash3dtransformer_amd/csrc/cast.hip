// bf16 copies of fp32 master weights for gfx950, several tensors in one launch, each optionally transposed as well.
//
// A training forward makes such copies of every parameter (the reference runs under autocast, which does the same), and the
// backward multiplies with the transposed weights.  Tensor by tensor these are launches of 2 to 5 us for a few KB each: 172
// casts and 53 transpositions, 0.72 ms of a 12.8 ms training step of the five-level model.  One launch per layer takes all
// of a layer's tensors: a workgroup owns one 64 x 64 tile of one of them, writes it as it is and, through LDS,
// transposed (55 launches, 0.27 ms; the step 12.75 -> 12.3 ms).  Bound by launch latency: 6 us for the six tensors of a
// 128-wide MLP, 10 for those of a 512-wide one (25 MB moved).
#include "f3d_device.h"
#include "f3d_internal.h"

namespace f3d {
namespace {

constexpr uint32_t kCastMax = 16, kCastTile = 64;

struct CastTable {
  const float* src[kCastMax];       // [rows][cols]
  uint16_t* dst[kCastMax];          // [rows][cols]
  uint16_t* dst_t[kCastMax];        // [cols][rows] or null
  uint32_t rows[kCastMax], cols[kCastMax], first[kCastMax];   // first workgroup of an entry
  uint32_t count;
};

__global__ __launch_bounds__(256) void cast_bf16_kernel(CastTable t) {
  __shared__ uint16_t s_tile[kCastTile][kCastTile + 2];
  uint32_t e = 0;
  while (e + 1 < t.count && blockIdx.x >= t.first[e + 1]) ++e;
  const uint32_t rows = t.rows[e], cols = t.cols[e], tile = blockIdx.x - t.first[e];
  const uint32_t tiles_c = (cols + kCastTile - 1) / kCastTile;
  const uint32_t r0 = tile / tiles_c * kCastTile, c0 = tile % tiles_c * kCastTile;
  const float* src = t.src[e];
  uint16_t* dst = t.dst[e];
  uint16_t* dst_t = t.dst_t[e];
  const uint32_t q = threadIdx.x / 16u, i4 = threadIdx.x % 16u * 4u;
  const bool vec = cols % 4u == 0u && ((uintptr_t)src & 15u) == 0u && ((uintptr_t)dst & 7u) == 0u;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t r = q + 16u * i, row = r0 + r, col = c0 + i4;
    uint16_t v[4] = {0, 0, 0, 0};
    if (row < rows) {
      const size_t at = (size_t)row * cols + col;
      if (vec && col < cols) {
        const float4 f = *reinterpret_cast<const float4*>(src + at);
        v[0] = float_to_bf16_bits(f.x); v[1] = float_to_bf16_bits(f.y);
        v[2] = float_to_bf16_bits(f.z); v[3] = float_to_bf16_bits(f.w);
        *reinterpret_cast<uint2*>(dst + at) = make_uint2(v[0] | ((uint32_t)v[1] << 16), v[2] | ((uint32_t)v[3] << 16));
      } else if (!vec) {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          if (col + j < cols) {
            v[j] = float_to_bf16_bits(src[at + j]);
            dst[at + j] = v[j];
          }
      }
    }
    if (dst_t) {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) s_tile[i4 + j][r] = v[j];
    }
  }
  if (!dst_t) return;
  __syncthreads();
  const bool vec_t = rows % 4u == 0u && ((uintptr_t)dst_t & 7u) == 0u;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t c = q + 16u * i, col = c0 + c, row = r0 + i4;
    if (col >= cols || row >= rows) continue;
    const size_t at = (size_t)col * rows + row;
    uint16_t v[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) v[j] = s_tile[c][i4 + j];
    if (vec_t) {
      *reinterpret_cast<uint2*>(dst_t + at) = make_uint2(v[0] | ((uint32_t)v[1] << 16), v[2] | ((uint32_t)v[3] << 16));
    } else {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j)
        if (row + j < rows) dst_t[at + j] = v[j];
    }
  }
}

}  // namespace
}  // namespace f3d

extern "C" int f3d_cast_bf16(const uint64_t* table, uint32_t count, int device, void* stream) {
  using namespace f3d;
  F3D_CHECK_ARG(count <= kCastMax, "at most %u tensors per call, got %u", kCastMax, count);
  F3D_CHECK_ARG(table || count == 0, "null table");
  CastTable t = {};
  uint64_t blocks = 0;
  for (uint32_t i = 0; i < count; ++i) {
    const uint64_t* e = table + 5 * i;
    if (e[3] == 0 || e[4] == 0) continue;
    F3D_CHECK_ARG(e[0] && e[1], "null tensor pointer in entry %u", i);
    F3D_CHECK_ARG(e[3] < (1ull << 31) && e[4] < (1ull << 31), "entry %u is too large", i);
    F3D_CHECK_ARG((e[0] & 3u) == 0 && (e[1] & 1u) == 0 && (e[2] & 1u) == 0, "entry %u is not aligned to its elements", i);
    const uint32_t n = t.count++;
    t.src[n] = reinterpret_cast<const float*>((uintptr_t)e[0]);
    t.dst[n] = reinterpret_cast<uint16_t*>((uintptr_t)e[1]);
    t.dst_t[n] = reinterpret_cast<uint16_t*>((uintptr_t)e[2]);
    t.rows[n] = (uint32_t)e[3];
    t.cols[n] = (uint32_t)e[4];
    t.first[n] = (uint32_t)blocks;
    blocks += (e[3] + kCastTile - 1) / kCastTile * ((e[4] + kCastTile - 1) / kCastTile);
    F3D_CHECK_ARG(blocks <= 0x7FFFFFull, "tensors too large for one launch");
  }
  if (blocks == 0) return F3D_OK;
  DeviceGuard guard(device);
  F3D_CHECK_ARG(guard.ok, "cannot select device %d", device);
  hipStream_t s = (hipStream_t)stream;
  SyncBracket sync(s);
  hipLaunchKernelGGL(cast_bf16_kernel, dim3((uint32_t)blocks), dim3(256), 0, s, t);
  F3D_CHECK_HIP(hipGetLastError());
  return F3D_OK;
}
