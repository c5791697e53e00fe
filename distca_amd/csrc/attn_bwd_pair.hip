// dQ and dK/dV of a batch of few blocks side by side.
//
// The backward's two kernels (attn_bwd_dq64_kernel.inc, attn_bwd_dkdv64_kernel.inc) depend on each other only through the row
// statistics that the dQ kernel makes on its way.  Where a batch has fewer blocks than the device has compute units, each kernel leaves most of
// it idle and lasts as long as its longest block, one after the other.  Here the launch that builds the lists makes the statistics as well
// (sched.hip, row_stats: a pass over dO and O, which at such sizes is nothing), and one launch takes both lists, dK/dV's, whose
// items are the longer ones, first.  389 tokens at 4/1 heads: the lists 9 us (statistics included), dQ 20 and dK/dV 23 one after the other; side by
// side 24.  The whole backward 56 -> 36 us there, 8 x 1000 tokens at 32/8 heads 299 -> 261, 8192 at 8/2 458 -> 395 (more at pair_backward, attn_cfg.h).
// dQ reads the statistics too, and O no more: 8 x 1000 tokens at 32/8 heads 269 -> 259 us, 20 x 300 134.5 -> 128.7, 2048 at 32/8 150 -> 146.5.
// Like the _split forms these park 20 to 40 registers in scratch memory, none of which comes back inside a loop over blocks or tiles.
#include "api_util.h"
#include "attn_bwd.h"
#include "attn_cfg.h"
#include "common.h"
#include "cut_blocks.h"

#include <type_traits>

namespace distca {
namespace {
namespace dq64 {
#define DQ64_BODY
#include "attn_bwd_dq64_kernel.inc"
}  // namespace dq64
namespace dkdv64 {
#define DKDV_BODY
#include "attn_bwd_dkdv64.h"
#define DKDV_SPLIT 1
#define DKDV_SHARED 0
#define DKDV_SEG 0
#define DKDV_NAME body
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SHARED
#undef DKDV_NAME
#define DKDV_SHARED 1
#define DKDV_NAME shared_body
#include "attn_bwd_dkdv64_kernel.inc"
#undef DKDV_SEG
#undef DKDV_NAME
#define DKDV_SEG 1
#define DKDV_NAME shards_body
#include "attn_bwd_dkdv64_kernel.inc"
}  // namespace dkdv64

constexpr int kPairLds = dq64::kLds > dkdv64::kLds ? dq64::kLds : dkdv64::kLds;
static_assert(dq64::kThreads == dkdv64::kThreads, "one launch");

// Workgroups 0 .. kv_groups - 1 are those over the dK/dV list, the others those over the dQ list.
__global__ __launch_bounds__(dq64::kThreads, 1) void ca_bwd_pair_kernel(BwdArgs kv, BwdArgs q, unsigned kv_groups) {
  if (blockIdx.x < kv_groups) dkdv64::body(kv, blockIdx.x);
  else dq64::dq64_body<false, false, true>(q, blockIdx.x - kv_groups);
}
__global__ __launch_bounds__(dq64::kThreads, 1) void ca_bwd_pair_shared_kernel(BwdArgs kv, BwdArgs q, unsigned kv_groups) {
  if (blockIdx.x < kv_groups) dkdv64::shared_body(kv, blockIdx.x);
  else dq64::dq64_body<false, false, true>(q, blockIdx.x - kv_groups);
}
__global__ __launch_bounds__(dq64::kThreads, 1) void ca_bwd_pair_shards_kernel(BwdArgs kv, BwdArgs q, unsigned kv_groups) {
  if (blockIdx.x < kv_groups) dkdv64::shards_body(kv, blockIdx.x);
  else dq64::dq64_body<true, false, true>(q, blockIdx.x - kv_groups);
}

// Adds up the pieces of both lists' blocks: parts 0 .. 2 kCutParts - 1 those of dK and dV, the others dQ's.  (One launch for both: us backward of
// 1500 tokens at 8/2 heads 59.4 -> 55.5, 2048 at 8/2 73 -> 69, 4096 at 4/1 101 -> 97.)
__global__ __launch_bounds__(kCutThreads) void ca_bwd_pair_combine_kernel(BwdArgs kv, BwdArgs q) {
  if (blockIdx.z < 2 * kCutParts) dkdv64::add_up_dkdv(kv, blockIdx.z);
  else dq64::add_up_dq(q, blockIdx.z - 2 * kCutParts);
}

}  // namespace

void DISTCA_FN(launch_pair_combine)(const BwdArgs &q, int64_t max_cut_q, const BwdArgs &kv, int64_t max_cut_kv, hipStream_t stream) {
  const int64_t most = max_cut_q > max_cut_kv ? max_cut_q : max_cut_kv;
  hipLaunchKernelGGL(ca_bwd_pair_combine_kernel, cut_grid(most, kv.hkv, 3 * kCutParts), dim3(kCutThreads), 0, stream, kv, q);
}

int DISTCA_FN(launch_pair)(const BwdArgs &q, int64_t grid_q, const BwdArgs &kv, int64_t grid_kv, bool shared, hipStream_t stream) {
  if (device_setup_pending(kSlotBwdPair)) {
    for (const void *kf : {(const void *)ca_bwd_pair_kernel, (const void *)ca_bwd_pair_shared_kernel, (const void *)ca_bwd_pair_shards_kernel})
      if (hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, kPairLds) != hipSuccess) return fail(DISTCA_E_LAUNCH, "ca_bwd: cannot reserve %d B of LDS", kPairLds);
    device_setup_done(kSlotBwdPair);
  }
  if (kv.shards.num_shards > 0 && !shared) return fail(DISTCA_E_INVALID, "ca_bwd: K/V shards in place need tasks over shared stored rows");
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)(grid_kv + grid_q)), dim3(dq64::kThreads), kPairLds, stream, kv, q, (unsigned)grid_kv); };
  if (kv.shards.num_shards > 0) launch(ca_bwd_pair_shards_kernel);
  else if (shared) launch(ca_bwd_pair_shared_kernel);
  else launch(ca_bwd_pair_kernel);
  return DISTCA_OK;
}

}  // namespace distca
