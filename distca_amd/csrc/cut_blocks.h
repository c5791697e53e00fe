// Adding up the pieces of cut blocks (sched.h, SplitTables).
#pragma once

#include "common.h"
#include "sched.h"

namespace distca {
// The kernels that add up the pieces of cut blocks have one text around what they add.  Grid: cut_grid(bound on cut blocks, kv heads, parts), each workgroup
// (256 threads) going through every gridDim.x-th cut block for one kv head and one of a block's 8 groups of 32 rows; wave w has d blocks 16 w .. 16 w + 15 and
// 64 + 16 w .. of those rows, in the accumulators' layout.  The sum leaves through LDS, whole rows in 16 byte stores: stored from there a store touched 32
// rows, 16 bytes of each.  us before (a wave going through the pieces one by one, stores from the accumulators' layout) -> after: dK/dV of 8192 tokens 38.0 ->
// 32.1 (33.5 with four pieces in flight alone), of 389 tokens at 4/1 heads 6.4 -> 4.1, forward of 4096 query rows at 8/2 heads over 32768 keys 17.0 -> 14.7;
// 4 is what the launch takes with nothing to add.
constexpr int kCutParts = 8, kCutThreads = 256;
inline dim3 cut_grid(int64_t max_cut, int hkv, int parts) {
  const int64_t most = (2048 / parts + hkv - 1) / hkv;   // workgroups beyond what runs at once only cost their start, also where little is cut
  return dim3((unsigned)(max_cut < most ? max_cut : most), hkv, parts);
}
// add(entry, o): adds the pieces of entry (unit, block, pieces, first slot) to o.  row_at(entry, r): where row r of the 32 goes, null if it does not exist.
template <class Add, class RowAt>
__device__ __forceinline__ void add_up_cut_blocks(const int32_t *cut, const int32_t *slot, Add add, RowAt row_at) {
  __shared__ __attribute__((aligned(16))) uint8_t rows[32 * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, g = lane >> 5;
  const int4 *entries = reinterpret_cast<const int4 *>(cut + 4);
  const int n = cut[0];
  int4 e = entries[first_cut_entry(cut, slot, blockIdx.x)];   // (asked for together with n)
  e.x = uniform_int(e.x), e.y = uniform_int(e.y), e.z = uniform_int(e.z), e.w = uniform_int(e.w);
  asm volatile("" : "+s"(e.x), "+s"(e.y), "+s"(e.z), "+s"(e.w));
  for (int c = blockIdx.x; c < n; c += gridDim.x) {
    if (c != (int)blockIdx.x) {
      e = entries[c];
      __syncthreads();  // the rows have left
    }
    f32x4 o[4] = {};
    add(e, o);
#pragma unroll
    for (int cq = 0; cq < 4; ++cq) {
      const int chunk = 2 * wave + 8 * (cq >> 1) + (cq & 1);
      *reinterpret_cast<elemx4 *>(rows + l32 * 256 + ((chunk ^ tile_swz(l32)) << 4) + 8 * g) = cvt4(o[cq][0], o[cq][1], o[cq][2], o[cq][3]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 16 * i + (tid >> 4);
      elem_t *at = row_at(e, r);
      if (at) *reinterpret_cast<elemx8 *>(at + 8 * (tid & 15)) = *reinterpret_cast<const elemx8 *>(rows + r * 256 + (((tid & 15) ^ tile_swz(r)) << 4));
    }
  }
}
// o += the pieces' sums in their order, four pieces' loads in flight at a time; piece j of this lane: first[j * step + k * pitch], k = 0 .. 3
__device__ __forceinline__ void add_pieces(const f32x4 *first, int64_t step, int pitch, int pieces, f32x4 (&o)[4]) {
  for (int j = 0; j < pieces; j += 4) {
    f32x4 v[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j + u < pieces) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[u][k] = first[(j + u) * step + k * pitch];
      }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j + u < pieces) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[k][r] += v[u][k][r];
      }
  }
}

}  // namespace distca
