// dK / dV of the varlen causal attention backward for gfx950, 64 keys per wave.
//
// One workgroup of 4 waves per (task, block of 256 keys, kv head), one wave per SIMD, so that a wave may use the
// SIMD's whole register file: the dK^T / dV^T accumulators of its 64 keys (4 sub-blocks of 16 keys x 8 blocks over d x 2
// matrices x 4 registers) fill the 256 accumulation registers, K of its keys stays in 64 vector registers as MFMA
// B operand, V of the workgroup's keys in LDS and three quarters of it (kVRegSlices) in registers too.  The query side (Q, dO and
// the row statistics of every head of the kv group, flattened into rows) streams through LDS in blocks of 32 rows, by LDS-direct loads into a ring of
// four stages, from the last block down to the first one the causal mask lets see these keys, or from that one up.
//
// With one wave per SIMD nothing else can use the SIMD's vector ALU while the wave waits for the matrix pipe, and
// a wave issues in order: an MFMA that finds the pipe busy holds up everything behind it.  So the arithmetic of a
// block (P = exp2(S c - lse2), dS = P (dP - delta), conversions to bf16) is written between the MFMAs of the same
// block, a few instructions behind each one, where it runs while the pipe works:
//
//   S  = Q K^T       32 MFMAs   A: rows of the Q tile (LDS), B: K registers
//   dP = dO V^T      32 MFMAs   A: rows of the dO tile, B: V (registers, LDS)            beside them: P from S
//   dV^T += dO^T P   32 MFMAs   A: transposing reads of the dO tile, B: P                beside them: dS from P, dP
//   dK^T += Q^T dS   32 MFMAs   A: transposing reads of the Q tile, B: dS
//
// Every LDS fragment a wave reads feeds four MFMAs (one per sub-block of the wave): half the LDS traffic per FLOP of
// a 32-key wave: with eight waves of 32 keys, two per SIMD, the LDS reads bounded the kernel.
//
// 16x16x32 MFMAs rather than 32x32x16, for the dQ kernel's reason (attn_bwd_dq64.hip): bound by power, and a FLOP of theirs moves half the
// accumulator bytes.  What they leave beside them, two issue slots each, is all used (240 other instructions beside a block's 128): on the way from
// one end of a document to the other four blocks, one per stage of the ring, make a round whose stages are constants in the reads' offsets, one wait
// does for the reads of eight MFMAs, and the diagonal's compares cover the half of the keys that it can touch.  The kernel, us, with 32x32x16 MFMAs ->
// with 16x16x32 -> with rounds and few waits (two boxes): 131072 packed tokens at 32/8 heads 23 250 -> 22 450 -> 21 020, a tick of 16384 tokens 2 575 ->
// 2 443 -> 2 328; documents of 128 to 2048 tokens 1 466 -> 1 429 -> 1 348, of 1024 (65536 tokens) 1 139 -> 1 098 -> 1 053, of 256 527 -> 506 -> 504;
// 389 tokens at 4/1 heads 28.5 -> 29.1 -> 28.9.  (With three lane-derived registers parked in scratch memory, reloaded ahead of each loop, where the
// reload waits for every request in flight: documents of 256 tokens 554, 389 tokens 30.8.)  The rounds and the bodies of masked and half blocks make
// 55 to 62 KB of code a form (40 to 45 before), within the 64 KB instruction cache of two compute units: 3 300 misses in 72 million requests of a launch over
// documents of 128 to 2048 tokens.
#include "api_util.h"
#include "attn_bwd.h"
#include "attn_cfg.h"
#include "common.h"
#include "cut_blocks.h"

#include <type_traits>

namespace distca {
namespace {

#include "attn_bwd_dkdv64.h"

#define DKDV_SHARED 0
#define DKDV_SEG 0
#define DKDV_SPLIT 0
#define DKDV_NAME ca_bwd_dkdv64_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SPLIT
#undef DKDV_NAME
#define DKDV_SPLIT 1
#define DKDV_NAME ca_bwd_dkdv64_split_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SHARED
#undef DKDV_NAME
#define DKDV_SHARED 1
#define DKDV_NAME ca_bwd_dkdv64_shared_split_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SEG
#undef DKDV_NAME
#define DKDV_SEG 1
#define DKDV_NAME ca_bwd_dkdv64_shards_split_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SPLIT
#undef DKDV_NAME
#define DKDV_SPLIT 0
#define DKDV_NAME ca_bwd_dkdv64_shards_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SEG
#undef DKDV_NAME
#define DKDV_SEG 0
#define DKDV_NAME ca_bwd_dkdv64_shared_kernel
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SHARED
#undef DKDV_SEG
#undef DKDV_SPLIT
#undef DKDV_NAME

__global__ __launch_bounds__(kCutThreads) void ca_bwd_dkdv64_combine_kernel(BwdArgs a) { add_up_dkdv(a, blockIdx.z); }

}  // namespace

#ifndef DISTCA_F16
int dkdv64_lds_bytes() { return kLds; }
#endif

void DISTCA_FN(launch_dkdv64_combine)(const BwdArgs &a, int64_t max_cut, hipStream_t stream) {
  hipLaunchKernelGGL(ca_bwd_dkdv64_combine_kernel, cut_grid(max_cut, a.hkv, 2 * kCutParts), dim3(kCutThreads), 0, stream, a);
}

int DISTCA_FN(launch_dkdv64)(const BwdArgs &a, int64_t grid, bool few, int64_t max_cut, bool shared, hipStream_t stream) {
  if (device_setup_pending(kSlotBwdLds64)) {
    const void *kernels[] = {(const void *)ca_bwd_dkdv64_kernel,        (const void *)ca_bwd_dkdv64_shared_kernel,       (const void *)ca_bwd_dkdv64_shards_kernel,
                             (const void *)ca_bwd_dkdv64_split_kernel,  (const void *)ca_bwd_dkdv64_shared_split_kernel, (const void *)ca_bwd_dkdv64_shards_split_kernel};
    for (const void *kf : kernels)
      if (hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess) return fail(DISTCA_E_LAUNCH, "ca_bwd: cannot reserve %d B of LDS", kLds);
    device_setup_done(kSlotBwdLds64);
  }
  if (a.shards.num_shards > 0 && !shared) return fail(DISTCA_E_INVALID, "ca_bwd: K/V shards in place need tasks over shared stored rows");
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kThreads), kLds, stream, a); };
  if (a.shards.num_shards > 0) launch(few ? ca_bwd_dkdv64_shards_split_kernel : ca_bwd_dkdv64_shards_kernel);
  else if (shared) launch(few ? ca_bwd_dkdv64_shared_split_kernel : ca_bwd_dkdv64_shared_kernel);
  else launch(few ? ca_bwd_dkdv64_split_kernel : ca_bwd_dkdv64_kernel);
  if (max_cut > 0) DISTCA_FN(launch_dkdv64_combine)(a, max_cut, stream);
  return DISTCA_OK;
}

}  // namespace distca
