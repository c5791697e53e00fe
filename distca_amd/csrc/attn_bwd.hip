// Varlen causal flash-attention backward (dQ, dK, dV) for gfx950.
//
// Stands where the reference calls flash-attn's varlen backward
// (distca/runtime/megatron/ops/fused_comm_attn.py:259-272).
//
// The backward runs as two kernels that both recompute P from (Q, K, LSE), so that neither
// needs floating-point atomics and the result is bit-reproducible (the `deterministic` switch
// of the reference's FlashAttnArgs holds by construction).  A single-kernel form that added
// dQ partial sums with fp32 atomics was measured first: the atomics alone (a 16 KB patch per
// 32 rows x 256 keys, 62 GB at 131 072 tokens, at the 1.3 TB/s the device adds floats at) took
// longer than the two kernels together.
//
//   1. ca_bwd_dq64_kernel (attn_bwd_dq64.hip): dQ, one workgroup of 4 waves per (task, block of 256 flattened
//      query rows, kv head), in the order of the forward tile schedule.  Its prologue, which reads a row's dO
//      anyway, also makes the row statistics both kernels need (delta = <dO, O>, lse * log2(e)) and leaves them in
//      the workspace.
//   2. ca_bwd_dkdv64_kernel (attn_bwd_dkdv64.hip): dK and dV, one workgroup of 4 waves per (task, block of
//      256 keys, kv head), in the order of the backward tile schedule.
//
// Batches of few blocks have both in one launch (attn_bwd_pair.hip; the rule: pair_backward).
#include "api_util.h"
#include "attn_bwd.h"
#include "attn_cfg.h"
#include "common.h"

#include <type_traits>

namespace distca {
namespace {

__global__ __launch_bounds__(256) void fill_zero_kernel(u32x4 *__restrict__ p, int64_t nvec) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (; i < nvec; i += stride) p[i] = u32x4{0, 0, 0, 0};
}

// How a backward is laid out in its workspace: the two lists, the row statistics, and, where blocks are cut into pieces, the lists'
// tables and the slots of both: side by side where they fit (slots_apart; attn_bwd_pair.hip writes both at a time), else in one place (dQ's
// pieces are then added up before the first of dK / dV is written).  In one place as well where the workspace has room for no more: what callers that
// keep a buffer sized it for before the slots lay side by side.
struct BwdLayout {
  int64_t sched_kv, sched_q, delta, lse2, tables_kv, tables_q, slots, slots_q, total;
  int64_t blocks_kv, blocks_q, items_kv, items_q;   // bounds on blocks, and room of the lists
  int32_t target_kv, target_q;                      // pieces aimed for per kv head, 0: whole blocks
  bool slots_apart;
};
// shared: tasks over shared stored rows (items are then over groups of tasks).  preferred: cut blocks of query rows as well, and
// key blocks whatever `deterministic` says.  one_place: the slots in one place.
BwdLayout bwd_layout(const distca_ca_params *p, bool shared, bool preferred, bool one_place = false) {
  BwdLayout w;
  w.blocks_kv = shared || preferred ? bwd_key_blocks_own_rows(p) : bwd_max_items(p) - bwd_split_target(p);
  w.blocks_q = dq_max_items(p);
  w.target_kv = preferred ? preferred_key_pieces(p) : bwd_split_target(p);
  w.target_q = preferred ? row_split_target(p, w.blocks_q, kCutFromTilesDq) : 0;
  w.items_kv = w.blocks_kv + w.target_kv;
  w.items_q = w.blocks_q + w.target_q;
  int64_t o = 0;
  auto take = [&](int64_t bytes) { const int64_t at = o; o = align_up(o + bytes, 256); return at; };
  w.sched_kv = take(sched_shared_region_bytes(p->num_tasks, w.items_kv));
  w.sched_q = take(sched_region_bytes(p->num_tasks, w.items_q));
  w.delta = take((int64_t)p->num_heads_q * p->total_q * 4);
  w.lse2 = take((int64_t)p->num_heads_q * p->total_q * 4);
  w.tables_kv = take(split_tables_bytes(w.blocks_kv, w.target_kv, w.items_kv));
  w.tables_q = take(split_tables_bytes(w.blocks_q, w.target_q, w.items_q));
  const int64_t kv = split_max_slots(w.blocks_kv, w.target_kv) * kDkdvSlotBytes, q = split_max_slots(w.blocks_q, w.target_q) * kDqSlotBytes;
  w.slots_apart = !one_place && slots_apart(p, w.blocks_kv, w.target_kv, w.blocks_q, w.target_q);
  w.slots = take((w.slots_apart || kv > q ? kv : q) * p->num_heads_kv);
  w.slots_q = w.slots_apart ? take(q * p->num_heads_kv) : w.slots;
  if (preferred && o > w.slots) take(256);   // (so that no call that brought the smallest workspace is taken for one that brought this)
  if (!preferred && bwd_small_pieces(p)) {
    const int64_t small = sched_shared_region_bytes(p->num_tasks, bwd_key_blocks_bound(p) + bwd_small_list_pieces(p)) +
                          sched_region_bytes(p->num_tasks, w.blocks_q) + 2 * align_up((int64_t)p->num_heads_q * p->total_q * 4, 256) + bwd_small_pieces_bytes(p);
    if (o < small) o = small;
  }
  w.total = o;
  return w;
}

// Whether dk or dv may lie on k or v: dense rows by their bytes; of shards in place only the buffers are known, which are then one.
bool gradients_on_inputs(const void *k, const void *v, const void *dk, const void *dv, int64_t bytes, bool shards) {
  const uintptr_t in[] = {(uintptr_t)k, (uintptr_t)v}, out[] = {(uintptr_t)dk, (uintptr_t)dv};
  for (uintptr_t i : in)
    for (uintptr_t o : out)
      if (shards ? i == o : i < o + (uintptr_t)bytes && o < i + (uintptr_t)bytes) return true;
  return false;
}

int grid_for(int64_t work_items) {
  int64_t g = (work_items + 255) / 256;
  const int64_t cap = (int64_t)num_compute_units() * 16;
  if (g > cap) g = cap;
  return g < 1 ? 1 : (int)g;
}

}  // namespace
}  // namespace distca

using namespace distca;

#ifndef DISTCA_F16
extern "C" int64_t distca_ca_bwd_workspace_bytes(const distca_ca_params *p) {
  if (!p) return fail(DISTCA_E_INVALID, "bwd_workspace_bytes: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  // the work lists and row statistics, and, for small batches whose caller does not ask for a deterministic backward, room for
  // the slots of a few pieces of key blocks
  return bwd_layout(p, false, false).total;
}

extern "C" int64_t distca_ca_bwd_workspace_preferred_bytes(const distca_ca_params *p) {
  if (!p) return fail(DISTCA_E_INVALID, "bwd_workspace_preferred_bytes: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  const int64_t own = bwd_layout(p, false, true).total, shared = bwd_layout(p, true, true).total, small = bwd_layout(p, false, false).total;
  return own > shared ? (own > small ? own : small) : (shared > small ? shared : small);
}

extern "C" int distca_ca_bwd(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse,
                             void *dq, void *dk, void *dv, const int32_t *cu_q, const int32_t *cu_k, const int32_t *kv_off,
                             const distca_ca_params *p, void *workspace, int64_t workspace_bytes, void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_bwd: null params");
  const int64_t row_bytes = (int64_t)p->num_heads_q * kHeadDim * 2;
  const BwdQuerySide qs{dout, q, out, lse, nullptr, nullptr, row_bytes, dq, nullptr, row_bytes};
  return (p->dtype == DISTCA_DTYPE_F16 ? run_bwd_f16 : run_bwd)(qs, k, v, dk, dv, cu_q, cu_k, kv_off, nullptr, p, workspace, workspace_bytes, stream);
}

extern "C" int distca_ca_bwd_tokens(const void *req_base, const int64_t *req_task_off, int64_t req_tok_bytes, const void *k,
                                    const void *v, void *dq_base, const int64_t *dq_task_off, int64_t dq_tok_bytes, void *dk,
                                    void *dv, const int32_t *cu_q, const int32_t *cu_k, const int32_t *kv_off,
                                    const distca_ca_params *p, void *workspace, int64_t workspace_bytes, void *stream) {
  return distca_ca_bwd_buffers(req_base, req_task_off, req_tok_bytes, k, v, nullptr, dq_base, dq_task_off, dq_tok_bytes, dk, dv, cu_q,
                               cu_k, kv_off, p, workspace, workspace_bytes, stream);
}

// kv_shards may be null here (distca_ca_bwd_tokens comes through this function); the public contract of the name
// requires it, which the header says.
extern "C" int distca_ca_bwd_buffers(const void *req_base, const int64_t *req_task_off, int64_t req_tok_bytes, const void *k,
                                     const void *v, const distca_kv_shards *kv_shards, void *dq_base, const int64_t *dq_task_off,
                                     int64_t dq_tok_bytes, void *dk, void *dv, const int32_t *cu_q, const int32_t *cu_k,
                                     const int32_t *kv_off, const distca_ca_params *p, void *workspace, int64_t workspace_bytes,
                                     void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_bwd: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  const int64_t row_bytes = (int64_t)p->num_heads_q * kHeadDim * 2, lse_bytes = (int64_t)p->num_heads_q * 4;
  if (lse_bytes & 15)
    return fail(DISTCA_E_UNSUPPORTED, "ca_bwd_tokens: %d query heads put the q part of a request token off 16-byte alignment", p->num_heads_q);
  // a server with no task this tick has empty offset arrays, which may come as null pointers; nothing reads them then
  if ((!req_task_off || !dq_task_off) && p->num_tasks > 0) return fail(DISTCA_E_INVALID, "ca_bwd_tokens: null offset array");
  if (req_tok_bytes < 3 * row_bytes + lse_bytes || (req_tok_bytes & 15))
    return fail(DISTCA_E_INVALID, "ca_bwd_tokens: request token of %lld B (needs >= %lld, multiple of 16)", (long long)req_tok_bytes, (long long)(3 * row_bytes + lse_bytes));
  if (dq_tok_bytes < row_bytes || (dq_tok_bytes & 15))
    return fail(DISTCA_E_INVALID, "ca_bwd_tokens: dq token of %lld B (needs >= %lld, multiple of 16)", (long long)dq_tok_bytes, (long long)row_bytes);
  const uint8_t *r = (const uint8_t *)req_base;
  // [dO | O | lse | q | pad]
  const BwdQuerySide qs{r, r ? r + 2 * row_bytes + lse_bytes : nullptr, r ? r + row_bytes : nullptr, nullptr,
                        r ? r + 2 * row_bytes : nullptr, req_task_off, req_tok_bytes, dq_base, dq_task_off, dq_tok_bytes};
  return (p->dtype == DISTCA_DTYPE_F16 ? run_bwd_f16 : run_bwd)(qs, k, v, dk, dv, cu_q, cu_k, kv_off, kv_shards, p, workspace, workspace_bytes, stream);
}
#endif  // !DISTCA_F16

namespace distca {
int DISTCA_FN(run_bwd)(const BwdQuerySide &qs, const void *k, const void *v, void *dk, void *dv, const int32_t *cu_q, const int32_t *cu_k,
                       const int32_t *kv_off, const distca_kv_shards *kv_shards, const distca_ca_params *p, void *workspace,
                       int64_t workspace_bytes, void *stream) {
  const void *dout = qs.dout, *q = qs.q, *out = qs.out;
  void *dq = qs.dq;
  if (!p) return fail(DISTCA_E_INVALID, "ca_bwd: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  const bool alias = kv_off != nullptr;
  if (!dout || !q || !k || !v || !out || (!qs.lse && !qs.lse_tok) || !dq || !dk || !dv || !cu_q || !cu_k) {
    if (p->num_tasks == 0 || (p->total_q == 0 && p->total_k == 0)) return DISTCA_OK;
    return fail(DISTCA_E_INVALID, "ca_bwd: null pointer");
  }
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || !aligned16(dout) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv))
    return fail(DISTCA_E_INVALID, "ca_bwd: tensors must be 16-byte aligned");
  // Tasks over shared K/V rows have one work item per (group of tasks, key block), or pieces of it.
  KvShards shards{};
  if (kv_shards) {
    rc = make_kv_shards(kv_shards, kv_off, true, &shards);
    if (rc) return rc;
  }
  const bool shared = alias;
  const bool roomy = workspace_bytes >= bwd_layout(p, shared, true).total;   // room for everything the call can use
  const bool preferred = roomy || workspace_bytes >= bwd_layout(p, shared, true, true).total;
  const BwdLayout w = bwd_layout(p, shared, preferred, !roomy);
  if (!workspace || workspace_bytes < w.total)
    return fail(DISTCA_E_WORKSPACE, "ca_bwd: workspace %lld B < required %lld B", (long long)workspace_bytes, (long long)w.total);
  if (!aligned16(workspace)) return fail(DISTCA_E_INVALID, "ca_bwd: workspace must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  uint8_t *ws = (uint8_t *)workspace;
  const int64_t kv_elems = (int64_t)p->total_k * p->num_heads_kv * kHeadDim;

  if (p->num_tasks == 0 || p->total_q == 0) {   // nothing to do but to clear dk and dv
    if (kv_elems > 0 && kv_shards)
      return fail(DISTCA_E_UNSUPPORTED, "ca_bwd_buffers: a batch without tasks or queries (there is nothing to tell which rows to clear)");
    if (kv_elems > 0) {
      hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(kv_elems / 8)), dim3(256), 0, s, (u32x4 *)dk, kv_elems / 8);
      hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(kv_elems / 8)), dim3(256), 0, s, (u32x4 *)dv, kv_elems / 8);
    }
    return check_launch("ca_bwd(clear)");
  }

  BwdArgs a;
  a.q = (const elem_t *)q; a.k = (const elem_t *)k; a.v = (const elem_t *)v; a.dout = (const elem_t *)dout;
  a.lse2 = (const float *)(ws + w.lse2); a.dscaled = (const float *)(ws + w.delta);
  a.lse2_w = (float *)(ws + w.lse2); a.dscaled_w = (float *)(ws + w.delta);
  a.out = (const elem_t *)out; a.lse = qs.lse; a.lse_tok = (const uint8_t *)qs.lse_tok;
  a.dq = (elem_t *)dq; a.dk = (elem_t *)dk; a.dv = (elem_t *)dv;
  a.qs_task_off = qs.task_off; a.qs_tok_bytes = qs.tok_bytes; a.dq_task_off = qs.dq_task_off; a.dq_tok_bytes = qs.dq_tok_bytes;
  a.cu_q = cu_q; a.cu_k = cu_k; a.kv_off = kv_off;
  a.grp_first = a.grp_tasks = a.grp_off = a.grp_lmax = nullptr;
  a.shards = shards;
  a.sched_items_off = (int32_t)sched_header_ints(p->num_tasks);
  a.hq = p->num_heads_q; a.hkv = p->num_heads_kv; a.group = p->num_heads_q / p->num_heads_kv;
  a.total_q = p->total_q; a.causal = p->causal != 0; a.scale = p->softmax_scale;
  a.group_magic = a.group == 1 ? 0u : (uint32_t)(((1ull << 32) + a.group - 1) / a.group);
  if ((uint64_t)p->max_seqlen_q * a.group * a.group >= (1ull << 32))
    return fail(DISTCA_E_UNSUPPORTED, "ca_bwd: max_seqlen_q * (Hq/Hkv)^2 must stay below 2^32");

  // ---- both work lists, and zeros where no work item writes dk / dv
  const bool few_q = few_row_blocks(p), few_kv = few_key_blocks(p, kSplitFewPerCU) || w.target_kv > 0;
  auto tables_of = [&](int64_t at, int64_t blocks, int32_t target) { return target > 0 ? split_tables(ws + at, blocks, target) : SplitTables{}; };
  // (dQ reads all of K and V, dK/dV each block's rows before it writes them: where the gradients take their inputs' place, dQ has to be done first)
  const bool pair = pair_backward(p, preferred) && (w.target_q == 0 || w.slots_apart) && !gradients_on_inputs(k, v, dk, dv, kv_elems * 2, kv_shards != nullptr);
  const ListJob q_list{cu_q, cu_k, launched_dq_geom(p, w.target_q), (int32_t *)(ws + w.sched_q), w.items_q, tables_of(w.tables_q, w.blocks_q, w.target_q)};
  const ListJob kv_list{cu_q, cu_k, launched_dkdv_geom(p, w.target_kv, preferred, shared, pair), (int32_t *)(ws + w.sched_kv), w.items_kv,
                        tables_of(w.tables_kv, w.blocks_kv, w.target_kv)};
  RowStats stats{};
  if (pair) stats = RowStats{(const uint8_t *)dout, (const uint8_t *)out, a.lse_tok, a.lse, a.qs_task_off, a.qs_tok_bytes, a.hq, a.total_q, kElemF16, a.lse2_w, a.dscaled_w};
  rc = launch_build_backward(kv_list, q_list, kv_off, p->num_tasks, BwdFill{(uint8_t *)dk, (uint8_t *)dv, (int64_t)p->num_heads_kv * kHeadDim * 2, p->total_k, shards}, stats, s);
  if (rc) return rc;

  // ---- dQ: one workgroup per (task, block of query rows, kv head).  It runs first: it also leaves the row
  // statistics (lse in the log2 domain, -delta) in the workspace, which the dK/dV kernel reads.  Side by side (attn_bwd_pair.hip) the launch
  // above has left them.
  BwdArgs aq;
  const int64_t grid_q = list_grid(p, w.items_q, few_q);
  {
    const int64_t grid = grid_q;
    if (grid > 0x7fffffff) return fail(DISTCA_E_INVALID, "ca_bwd: grid too large");
    a.merge_tiles = q_list.geom.merge_tiles;
    a.sched = q_list.ws;
    a.zero_row = ws + w.sched_q + sched_zero_row_off(p->num_tasks, w.items_q);
    a.tickets = (int32_t *)(ws + w.sched_q + sched_ticket_off(p->num_tasks, w.items_q));
    a.cut = q_list.split.cut; a.slot = q_list.split.slot;
    a.partial = ws + w.slots_q;
    aq = a;
    if (!pair) {
      ScopedTimer timer(DISTCA_TIMER_CA_BWD_DQ, s);
      rc = DISTCA_FN(launch_dq64)(a, grid, few_q, w.target_q > 0 ? split_max_cut(w.blocks_q, w.target_q) : 0, s);
      if (rc) return rc;
    }
  }
  // ---- dK, dV: one workgroup per (task, 256-key block, kv head)
  {
    // items tile stored rows (tasks that own their rows, or groups of tasks that share them); the list may have more room
    const int64_t grid = list_grid(p, bwd_key_blocks_own_rows(p) + w.target_kv, few_kv);
    if (grid > 0x7fffffff) return fail(DISTCA_E_INVALID, "ca_bwd: grid too large");
    if (shared) {
      const SharedGroups sg = shared_groups(kv_list.ws, p->num_tasks, w.items_kv);
      a.grp_first = sg.first; a.grp_tasks = sg.tasks; a.grp_off = sg.off; a.grp_lmax = sg.lmax;
    }
    a.sched = kv_list.ws;
    a.zero_row = ws + w.sched_kv + sched_zero_row_off(p->num_tasks, w.items_kv);
    a.tickets = (int32_t *)(ws + w.sched_kv + sched_ticket_off(p->num_tasks, w.items_kv));
    a.cut = kv_list.split.cut; a.slot = kv_list.split.slot;
    a.partial = ws + w.slots;
    ScopedTimer timer(DISTCA_TIMER_CA_BWD, s);
    const int64_t max_cut = w.target_kv > 0 ? split_max_cut(w.blocks_kv, w.target_kv) : 0;
    if (pair) {
      rc = DISTCA_FN(launch_pair)(aq, grid_q, a, grid, shared, s);
      if (rc) return rc;
      if (w.target_q > 0 && max_cut > 0) DISTCA_FN(launch_pair_combine)(aq, split_max_cut(w.blocks_q, w.target_q), a, max_cut, s);
      else if (max_cut > 0) DISTCA_FN(launch_dkdv64_combine)(a, max_cut, s);
    } else {
      rc = DISTCA_FN(launch_dkdv64)(a, grid, few_kv, max_cut, shared, s);
      if (rc) return rc;
    }
  }
  return check_launch("ca_bwd");
}
}  // namespace distca
