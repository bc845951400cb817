// Streamed tiles: what the forward (fwd_stream.hip) and the backward
// (bwd_stream.hip) of the same shapes share.
#pragma once

#include "common.h"
#include "params.h"

namespace farope {

constexpr int kStreamNW = 4;                  // waves per workgroup, 32 rows each (16 in 64-row tiles)
static_assert(32 * kStreamNW == kStreamTileRows && 64 * kStreamNW == kStreamThreads, "");
constexpr int kStageRows = 64;                // streamed rows per stage

// Element offset of (row, column) in an unpadded tile whose 16-byte chunks
// are XOR-swizzled per row with period 16: 16-byte reads of 16 consecutive
// rows and transposed reads of rows 4lg + e are free of bank conflicts.
template <int D> __device__ __forceinline__ int swz_chunk(int r) {
  if constexpr (D == 128)  // (the low chunk bit stays: rows of 16 chunks cover all banks)
    return ((r >> 1) & 7) << 1;
  else if constexpr (D == 64)
    return ((((r >> 1) & 3) ^ ((r >> 2) & 2)) << 1) | ((r >> 3) & 1);
  else
    return (r >> 2) & 3;
}
template <int D> __device__ __forceinline__ int swz(int r, int col) {
  return r * D + (((col >> 3) ^ swz_chunk<D>(r)) << 3) + (col & 7);
}

// 4 bytes per lane from a buffer straight into LDS (lane l lands at lds + 4 l).
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t r, void* lds, unsigned voff, unsigned soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, voff, soff, 0, 0);
}

// Barrier between stages: this wave's LDS loads have landed (the fence of
// lds_barrier does not cover them on every path) and its LDS reads are done.
__device__ __forceinline__ void stage_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  lds_barrier();
}

// One stage of a streamed tensor.  A 16-byte-per-lane load fills 64 * 8 / D
// consecutive rows: lane l lands at row l / (D/8), chunk slot l % (D/8), so it
// fetches the chunk whose swizzled place that slot is.
template <int D> struct StreamSrc {
  static constexpr int CPR = D / 8, RPI = 64 / CPR, GROUPS = kStageRows / RPI;
  __amdgpu_buffer_rsrc_t rs;
  unsigned voff;      // this lane's byte offset in rows 0 .. of the wave's first group
  unsigned row_b;     // bytes between rows
  __device__ __forceinline__ void init(const void* base, int64_t stride, int N, int wave, int lane) {
    rs = make_rsrc(base, (unsigned)(((int64_t)(N - 1) * stride + D) * 2));
    row_b = (unsigned)((int)stride * 2);
    const int r = wave * RPI + lane / CPR;
    voff = (unsigned)r * row_b + (unsigned)(((lane % CPR) ^ swz_chunk<D>(r)) * 16);
  }
  template <typename S> __device__ __forceinline__ void load(S* dst, int wave, int row0) const {
#pragma unroll
    for (int g = 0; g < GROUPS / kStreamNW; ++g)
      lds_dma16(rs, dst + (wave + g * kStreamNW) * RPI * D, voff, (unsigned)(row0 + g * kStreamNW * RPI) * row_b);
  }
};

}  // namespace farope
