// dQ of the varlen causal attention backward for gfx950, 64 query rows per wave.
//
// One workgroup of 4 waves per (task, block of 256 flattened query rows, kv head), one wave per SIMD with the
// SIMD's whole register file.  A wave owns four sub-blocks of 16 rows: their Q and dO stay in registers as MFMA B
// operands, their dQ^T accumulators in the accumulation registers.  K/V tiles of 32 keys stream through a ring of
// four LDS stages by LDS-direct loads, from key 0 up to the last key the block's rows see; every LDS fragment a
// wave reads (K rows, V rows, transposed K) feeds four MFMAs, one per sub-block.  With one wave per SIMD the
// arithmetic of a tile is written between the MFMAs of the same tile:
//
//   S^T  = K Q^T        32 MFMAs   A: rows of the K tile (LDS), B: Q registers
//   dP^T = V dO^T       32 MFMAs   A: rows of the V tile, B: dO registers
//   dQ^T += K^T dS^T    32 MFMAs   A: transposing reads of the K tile, B: dS = P (dP - delta) with P = exp2(S c - lse2)
//
// 16x16x32 MFMAs rather than 32x32x16: the kernel is bound by power, and a FLOP of theirs moves half the accumulator
// bytes (and twice the operand bytes, which cost less where neighbours share one).  A loop of nothing but MFMAs (probe.hip)
// delivers 1 800 to 1 880 TFLOP/s with the latter and 1 960 to 2 080 with the former, with half a KB of LDS reads and three vector instructions per
// 32 K FLOP beside them 1 570 to 1 640 and 1 700 to 1 780 (by box).  They leave 2 issue slots each for anything else (the larger ones 5), so the side work
// is spread over the whole tile.  The kernel, before -> after: 131072 packed tokens at 32/8 heads 16 870 us -> 15 510
// (1.66 -> 1.81 GHz at 79 % of the pipe's cycles), a tick of 16384 tokens 1 837 -> 1 711, documents of 128 to 2048 tokens 1 268 -> 1 251.
//
// The prologue also makes the row statistics of the backward (delta = <dO, O>, lse in the log2 domain) and leaves
// them in the workspace for the dK/dV kernel, which runs after this one.
#include "api_util.h"
#include "attn_bwd.h"
#include "attn_cfg.h"
#include "common.h"
#include "cut_blocks.h"

#include <type_traits>

namespace distca {
namespace {

#include "attn_bwd_dq64_kernel.inc"

__global__ __launch_bounds__(kCutThreads) void ca_bwd_dq64_combine_kernel(BwdArgs a) { add_up_dq(a, blockIdx.z); }

}  // namespace

void DISTCA_FN(launch_dq64_combine)(const BwdArgs &a, int64_t max_cut, hipStream_t stream) {
  hipLaunchKernelGGL(ca_bwd_dq64_combine_kernel, cut_grid(max_cut, a.hkv, kCutParts), dim3(kCutThreads), 0, stream, a);
}

int DISTCA_FN(launch_dq64)(const BwdArgs &a, int64_t grid, bool few, int64_t max_cut, hipStream_t stream) {
  if (device_setup_pending(kSlotBwdDq64)) {
    const void *kernels[] = {(const void *)ca_bwd_dq64_kernel<false, false, false>, (const void *)ca_bwd_dq64_kernel<true, false, false>,
                             (const void *)ca_bwd_dq64_kernel<false, true, false>,  (const void *)ca_bwd_dq64_kernel<true, true, false>,
                             (const void *)ca_bwd_dq64_kernel<false, false, true>,  (const void *)ca_bwd_dq64_kernel<true, false, true>};
    for (const void *kf : kernels) {
      hipError_t e = hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
      if (e != hipSuccess) return fail(DISTCA_E_LAUNCH, "ca_bwd: cannot reserve %d B of LDS: %s", kLds, hipGetErrorString(e));
    }
    device_setup_done(kSlotBwdDq64);
  }
  const dim3 g((unsigned)grid), b(kThreads);
  const bool seg = a.shards.num_shards > 0;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, kLds, stream, a); };
  if (few) launch(seg ? ca_bwd_dq64_kernel<true, false, true> : ca_bwd_dq64_kernel<false, false, true>);
  else if (a.merge_tiles > 0) launch(seg ? ca_bwd_dq64_kernel<true, true, false> : ca_bwd_dq64_kernel<false, true, false>);
  else launch(seg ? ca_bwd_dq64_kernel<true, false, false> : ca_bwd_dq64_kernel<false, false, false>);
  if (max_cut > 0) DISTCA_FN(launch_dq64_combine)(a, max_cut, stream);
  return DISTCA_OK;
}

}  // namespace distca
