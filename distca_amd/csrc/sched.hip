// Device builder and host mirror of the tile schedule described in sched.h.
#include <algorithm>
#include <vector>

#include "api_util.h"
#include "attn_cfg.h"
#include "common.h"
#include "kv_shards.h"
#include "sched.h"

namespace distca {
namespace {

constexpr int kSchedThreads = 1024;
// Batches of at most this many tasks (nearly all of them) are worked on in LDS: the builder is one workgroup whose phases are
// chains of dependent reads, and at half a microsecond a read from memory they were most of its time.
constexpr int kLdsTasks = kSchedThreads;

__device__ __forceinline__ int32_t block_inclusive_scan_i32(int32_t v, int32_t *wave_sums) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_inclusive_scan_i32(v);
  __syncthreads();
  if (lane == 63) wave_sums[wave] = v;
  __syncthreads();
  // (the sums of the waves before this one: a read and a scan instead of a chain of up to fifteen reads)
  const int32_t sum = wave_inclusive_scan_i32(lane < kSchedThreads / 64 ? wave_sums[lane] : 0);
  return v + (wave > 0 ? __builtin_amdgcn_readlane(sum, __builtin_amdgcn_readfirstlane(wave) - 1) : 0);
}

// The task bounds as the builder reads them: in LDS when they fit.
struct Tasks {
  const int32_t *cu_q, *cu_k, *kv_off;
  int32_t n;
  __device__ __forceinline__ int32_t lq(int32_t b) const { return cu_q[b + 1] - cu_q[b]; }
  __device__ __forceinline__ int32_t lk(int32_t b) const { return cu_k[b + 1] - cu_k[b]; }
};
struct TaskCache {
  int32_t q[kLdsTasks + 1], k[kLdsTasks + 1], off[kLdsTasks];
};
__device__ __forceinline__ Tasks load_tasks(TaskCache &c, const int32_t *cu_q, const int32_t *cu_k, const int32_t *kv_off, int32_t n) {
  if (n > kLdsTasks) return Tasks{cu_q, cu_k, kv_off, n};
  for (int i = threadIdx.x; i <= n; i += kSchedThreads) {
    c.q[i] = cu_q[i];
    c.k[i] = cu_k[i];
    if (kv_off && i < n) c.off[i] = kv_off[i];
  }
  __syncthreads();
  return Tasks{c.q, c.k, c.off, n};
}

// What the list is made over.  TaskUnits: every task has its own blocks (query blocks in the forward and dQ lists, key
// blocks in the dK/dV list).  GroupUnits (the dK/dV list when tasks share stored K/V rows): a unit is a group of tasks
// that read prefixes of one stored document, its blocks are the document's key blocks, and a block's cost is the sum
// over the group's tasks of the query blocks that see it -- one work item owns a key block's dK/dV on behalf of every
// task, so that the sums need neither atomics nor a fixed-up order.
template <bool BWD>
struct TaskUnits {
  Tasks t;
  SchedGeom g;
  __device__ __forceinline__ int32_t blocks(int32_t b) const {
    const int32_t n = BWD ? bwd_num_blocks(g, t.lq(b), t.lk(b)) : fwd_num_items(g, t.lq(b), t.lk(b));
    return n < 0 ? 0 : n;
  }
  __device__ __forceinline__ int32_t cost(int32_t b, int32_t i) const {
    return BWD ? bwd_cost(g, t.lq(b), t.lk(b), i) : fwd_item_cost(g, t.lq(b), t.lk(b), i);
  }
};
struct GroupUnits {
  Tasks t;
  SchedGeom g;
  const int32_t *grp_first, *grp_tasks, *grp_lmax;
  __device__ __forceinline__ int32_t blocks(int32_t u) const { return ceil_div_pow2(grp_lmax[u], g.kv_per_block); }
  __device__ __forceinline__ int32_t cost(int32_t u, int32_t i) const {
    int32_t c = 0;
    for (int32_t e = grp_first[u]; e < grp_first[u + 1]; ++e) {
      const int32_t b = grp_tasks[e], lk = t.lk(b);
      if (i * g.kv_per_block < lk) c += bwd_cost(g, t.lq(b), lk, i);
    }
    return c;
  }
};

// Largest b in [0, B) with base[b] <= e.
__device__ __forceinline__ int32_t find_task(const int32_t *base, int32_t num_tasks, int32_t e) {
  int32_t lo = 0, hi = num_tasks;  // invariant: base[lo] <= e < base[hi]
  while (hi - lo > 1) {
    int32_t mid = (lo + hi) >> 1;
    if (base[mid] <= e) lo = mid; else hi = mid;
  }
  return lo;
}

struct ListScratch {
  int32_t bins[kSchedBins], base[kLdsTasks + 1], wave_sums[kSchedThreads / 64], ranked[4];
  uint32_t order[kLdsTasks];   // of a dK/dV list's entries: (unit, block, piece), as one number
  int32_t carry, num_cut, num_slots, piece;
  unsigned long long total_cost;
};

// The sorted list over `num_units` units.  `hdr_units` sizes the header (the task count, whatever the units are).
// `split`: where the tables of a list with cut blocks go (null arrays when nothing is cut).
template <bool BWD, class Units>
__device__ __forceinline__ void build_list(ListScratch &s, const Units &u, int32_t num_units, int32_t hdr_units, const SchedGeom &g,
                                           int32_t *__restrict__ ws, int32_t max_items, const SplitTables &split) {
  int32_t *items = ws + sched_header_ints(hdr_units);
  const int tid = threadIdx.x;
  int32_t *base = num_units <= kLdsTasks ? s.base : ws + 4;

  // 1. exclusive prefix of block counts per unit
  for (int i = tid; i < kSchedBins; i += kSchedThreads) s.bins[i] = 0;
  if (tid == 0) s.total_cost = 0, s.num_cut = s.num_slots = 0;
  if (tid < 4) s.ranked[tid] = 0;
  int32_t running = 0;
  for (int32_t c0 = 0; c0 < num_units; c0 += kSchedThreads) {
    const int32_t b = c0 + tid;
    const int32_t n = b < num_units ? u.blocks(b) : 0;
    const int32_t incl = block_inclusive_scan_i32(n, s.wave_sums);
    if (b < num_units) base[b] = ws[4 + b] = running + incl - n;
    if (tid == kSchedThreads - 1) s.carry = running + incl;
    __syncthreads();
    running = s.carry;
  }
  // (a list with pieces has room for split_target more than its blocks; sizes that understate the batch drop whole blocks)
  const int32_t max_blocks = max_items - (g.split_target > 0 ? g.split_target : 0);
  const int32_t nitems = running < max_blocks ? running : max_blocks;
  if (tid == 0) base[num_units] = ws[4 + num_units] = running;
  __syncthreads();

  // The first blocks of every thread are found once and kept: (unit, block, cost).
  constexpr int kKept = 2;
  int32_t unit[kKept], block[kKept], price[kKept];
#pragma unroll
  for (int c = 0; c < kKept; ++c) {
    const int32_t e = tid + c * kSchedThreads;
    unit[c] = block[c] = price[c] = 0;
    if (e < nitems) {
      unit[c] = find_task(base, num_units, e);
      block[c] = e - base[unit[c]];
      price[c] = u.cost(unit[c], block[c]);
    }
  }
  auto each_block = [&](auto f) {
#pragma unroll
    for (int c = 0; c < kKept; ++c)
      if (tid + c * kSchedThreads < nitems) f(unit[c], block[c], price[c]);
    for (int32_t e = tid + kKept * kSchedThreads; e < nitems; e += kSchedThreads) {
      const int32_t b = find_task(base, num_units, e);
      f(b, e - base[b], u.cost(b, e - base[b]));
    }
  };

  // 1b. (when asked for) the piece size that cuts expensive blocks
  int32_t piece = 0;
  if (g.split_target > 0) {
    unsigned long long local = 0;
    each_block([&](int32_t, int32_t, int32_t cost) { local += (unsigned long long)cost; });
    // (three sums that cannot overflow: a thread's costs stay below 2^58)
    const int32_t lo = wave_inclusive_scan_i32((int32_t)(local & 0xffff)), mid = wave_inclusive_scan_i32((int32_t)((local >> 16) & 0xffff)),
                  hi = wave_inclusive_scan_i32((int32_t)(local >> 32));
    if ((tid & 63) == 63) atomicAdd(&s.total_cost, (unsigned long long)(uint32_t)lo + ((unsigned long long)(uint32_t)mid << 16) + ((unsigned long long)(uint32_t)hi << 32));
    if (tid == 0) s.piece = 0;
    __syncthreads();
    if (tid == 0) s.piece = piece_size(s.total_cost, g.split_target, g.min_piece);
    __syncthreads();
    piece = s.piece;
  }

  // 2. histogram of cost bins, blocks cut into pieces of at most `size` (0: whole)
  const bool fixed = g.units_per_head > 0;   // fixed pieces (or none), not equal parts
  auto histogram = [&](int32_t size) {
    each_block([&](int32_t, int32_t, int32_t cost) {
      if (fixed) {
        const int32_t k = fixed_piece_count(cost, size);
        if (k > 1) atomicAdd(&s.bins[cost_bin(g, size)], k - 1);
        atomicAdd(&s.bins[cost_bin(g, cost - (k - 1) * size)], 1);
        return;
      }
      const int32_t k = piece_count(cost, size);
      for (int32_t j = 0; j < k; ++j) atomicAdd(&s.bins[cost_bin(g, piece_begin(cost, j + 1, k) - piece_begin(cost, j, k))], 1);
    });
    __syncthreads();
  };
  // 3. start offset of each bin when bins are laid out from the most expensive down; `look` sees every bin's start and count
  auto offsets = [&](auto look) {
    constexpr int kPer = kSchedBins / kSchedThreads;
    int32_t cnt[kPer], local = 0;
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
      cnt[v] = s.bins[kSchedBins - 1 - (tid * kPer + v)];
      local += cnt[v];
    }
    const int32_t incl = block_inclusive_scan_i32(local, s.wave_sums);
    int32_t start = incl - local;
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
      const int bin = kSchedBins - 1 - (tid * kPer + v);
      s.bins[bin] = look(bin, start, cnt[v]);
      start += cnt[v];
    }
    __syncthreads();
  };
  auto starts = [](int, int32_t start, int32_t) { return start; };
  histogram(fixed ? 0 : piece);
  if (fixed) {
    // whole blocks first: their costs by rank decide whether, and how finely, blocks are cut
    offsets([&](int bin, int32_t start, int32_t n) {
      for (int k = 0; k < 4; ++k) {
        const int64_t rank = (int64_t)k * g.units_per_head;
        if (start <= rank && rank < start + n) s.ranked[k] = bin << g.cost_shift;
      }
      return n;
    });
    if (tid < 64) {   // a lane per size
      const int32_t least = piece;
      int32_t size;
      float t = pieces_time(g, (float)s.total_cost, nitems, s.ranked[0], least, (tid % kPieceTries) + 1, &size);
#pragma unroll
      for (int off = kPieceTries / 2; off > 0; off >>= 1) {
        const float to = __shfl_xor(t, off, 64);
        const int32_t so = __shfl_xor(size, off, 64);
        if (to < t || (to == t && so > size)) t = to, size = so;
      }
      if (tid == 0) s.piece = t < worth_cutting(g) * whole_time(g, (float)s.total_cost, nitems, s.ranked) ? size : 0;
    }
    __syncthreads();
    piece = s.piece;
    if (piece > 0) {
      for (int i = tid; i < kSchedBins; i += kSchedThreads) s.bins[i] = 0;
      __syncthreads();
      histogram(piece);
    }
  }
  offsets(starts);

  // (piece numbers are below kMaxPieces)
  auto order_of = [](int32_t block, int32_t piece) { return ((uint32_t)block << 6) | (uint32_t)piece; };
  // 4. scatter
  each_block([&](int32_t b, int32_t i, int32_t cost) {
    const int32_t k = fixed ? fixed_piece_count(cost, piece) : piece_count(cost, piece);
    int32_t slot = -1;
    if (k > 1 && split.cut) {
      slot = atomicAdd(&s.num_slots, k);
      reinterpret_cast<int4 *>(split.cut + 4)[atomicAdd(&s.num_cut, 1)] = make_int4(b, i, k, slot);
    }
    int32_t run = fixed && k > 1 ? atomicAdd(&s.bins[cost_bin(g, piece)], k - 1) : 0;   // places of the block's full pieces
    for (int32_t j = 0; j < k; ++j) {
      int32_t cj, pos;
      if (fixed) {
        cj = j < k - 1 ? piece : cost - (k - 1) * piece;
        pos = j < k - 1 ? run++ : atomicAdd(&s.bins[cost_bin(g, cj)], 1);
      } else {
        cj = piece_begin(cost, j + 1, k) - piece_begin(cost, j, k);
        pos = atomicAdd(&s.bins[cost_bin(g, cj)], 1);
      }
      if (pos < max_items) {
        reinterpret_cast<int4 *>(items)[pos] = make_int4(b, i, cj, j | (k << 16));
        if (split.cut) reinterpret_cast<int2 *>(split.slot)[pos] = make_int2(slot < 0 ? -1 : slot + j, cost);
        if (BWD && pos < kLdsTasks) s.order[pos] = order_of(base[b] + i, j);
      }
    }
  });
  __syncthreads();
  // after the scatter the counter of the cheapest bin holds the number of entries
  const int32_t entries = s.bins[0], total = entries < max_items ? entries : max_items;
  // 5. (backward) walk direction by rank.  The scatter above puts the entries of one cost bin in whatever order
  // the threads came; an entry's rank in the order (bin, unit, block, piece) is the start of its bin plus the
  // number of entries of the bin that precede it in that order, counted here, and is the same in every run.
  // (A list of one round has no upward walks.)
  if (BWD && g.walk_round > 0 && total > g.walk_round) {
    for (int32_t pos = tid; pos < total; pos += kSchedThreads) {
      const int4 it = reinterpret_cast<const int4 *>(items)[pos];
      const int32_t bin = cost_bin(g, it.z);
      const int32_t seg0 = bin == kSchedBins - 1 ? 0 : s.bins[bin + 1];  // bins lie from the most expensive down
      const int32_t seg1 = s.bins[bin] < total ? s.bins[bin] : total;
      const int64_t key = ((int64_t)(base[it.x] + it.y) << 16) | item_piece(it.w);
      int32_t rank = seg0;
      if (seg1 - seg0 <= kWalkTieLimit) {
        if (total <= kLdsTasks && nitems <= kLdsTasks) {   // from LDS: 76 items of 8192 tokens, 5.7 us of the launch's 24 otherwise
          const uint32_t mine = order_of(base[it.x] + it.y, item_piece(it.w));
          for (int32_t o = seg0; o < seg1; ++o) rank += s.order[o] < mine;
        } else {
          for (int32_t o = seg0; o < seg1; ++o) {
            const int4 ot = reinterpret_cast<const int4 *>(items)[o];
            rank += (((int64_t)(base[ot.x] + ot.y) << 16) | item_piece(ot.w)) < key;
          }
        }
      }
      // only the flag bit changes, and the reads above look at the other bits only
      if ((rank / g.walk_round) & 1) items[4 * pos + 3] = it.w | kWalkUp;
    }
  }
  if (tid == 0) {
    ws[0] = total;
    ws[1] = running;
    // entries that found no room in the list (blocks beyond max_items count whole): never 0 < by construction
    // when the caller's sizes bound its sequence lengths; tests and debugging read it
    ws[2] = (entries > max_items ? entries - max_items : 0) + (running > max_blocks ? running - max_blocks : 0);
    if (split.cut) split.cut[0] = s.num_cut, split.cut[1] = s.num_slots, split.cut[2] = fixed ? piece : 0;
  }
  if (tid < kZeroRowBytes / 4) ws[sched_zero_row_off(hdr_units, max_items) / 4 + tid] = 0;
  if (tid < kTicketBytes / 4) ws[sched_ticket_off(hdr_units, max_items) / 4 + tid] = 0;
}

template <bool BWD>
__device__ __forceinline__ void build_own(ListScratch &s, TaskCache &cache, const ListJob &j, int32_t num_tasks) {
  const TaskUnits<BWD> u{load_tasks(cache, j.cu_q, j.cu_k, nullptr, num_tasks), j.geom};
  build_list<BWD>(s, u, num_tasks, num_tasks, j.geom, j.ws, (int32_t)j.max_items, j.split);
  if (threadIdx.x == 0) j.ws[3] = 0;
}
__global__ __launch_bounds__(kSchedThreads) void build_forward_kernel(ListJob j, int32_t num_tasks) {
  __shared__ ListScratch s;
  __shared__ TaskCache cache;
  build_own<false>(s, cache, j, num_tasks);
}

// The dK/dV list over tasks that share stored K/V rows (see GroupUnits and, for the arrays, SharedGroups in sched.h).
// Tasks with queries form a group when they start at the same stored row.  Quadratic in the task count where a task
// looks for its group (a thousand tasks: a thousand comparisons per thread).
struct GroupScratch {
  int32_t first[kLdsTasks + 1], tasks[kLdsTasks], off[kLdsTasks], lmax[kLdsTasks], lead[kLdsTasks], gid[kLdsTasks];
  int32_t carry, violations;
};
__device__ void build_shared(ListScratch &s, TaskCache &cache, GroupScratch &gs, const ListJob &j, const int32_t *kv_off, int32_t num_tasks,
                             int32_t total_k) {
  const SharedGroups out = shared_groups(j.ws, num_tasks, j.max_items);
  const Tasks t = load_tasks(cache, j.cu_q, j.cu_k, kv_off, num_tasks);
  const bool fits = num_tasks <= kLdsTasks;
  SharedGroups sg = out;
  int32_t *lead = out.tmp, *gid = out.tmp + num_tasks;
  if (fits) sg.first = gs.first, sg.tasks = gs.tasks, sg.off = gs.off, sg.lmax = gs.lmax, lead = gs.lead, gid = gs.gid;
  const int tid = threadIdx.x;
  auto live = [&](int32_t b) { return t.lq(b) > 0 && t.lk(b) > 0; };
  if (tid == 0) gs.violations = 0;
  // a. the first live task that starts where task b starts
  for (int32_t b = tid; b < num_tasks; b += kSchedThreads) {
    int32_t l = -1;
    if (live(b)) {
      const int32_t off = t.kv_off[b];
      for (l = 0; l < b; ++l)
        if (t.kv_off[l] == off && live(l)) break;
    }
    lead[b] = l;
  }
  for (int32_t u = tid; u <= num_tasks; u += kSchedThreads) {
    sg.first[u] = 0;
    if (u < num_tasks) sg.lmax[u] = 0;
  }
  __syncthreads();
  // b. groups numbered in the order of their first tasks
  int32_t ngroups = 0;
  for (int32_t c0 = 0; c0 < num_tasks; c0 += kSchedThreads) {
    const int32_t b = c0 + tid;
    const int32_t is_lead = b < num_tasks && lead[b] == b ? 1 : 0;
    const int32_t incl = block_inclusive_scan_i32(is_lead, s.wave_sums);
    if (is_lead) gid[b] = ngroups + incl - 1;
    if (tid == kSchedThreads - 1) gs.carry = ngroups + incl;
    __syncthreads();
    ngroups = gs.carry;
  }
  __syncthreads();
  // c. members, longest prefix and first row of every group
  for (int32_t b = tid; b < num_tasks; b += kSchedThreads)
    if (lead[b] >= 0) {
      const int32_t u = gid[lead[b]];
      atomicAdd(&sg.first[u + 1], 1);
      atomicMax(&sg.lmax[u], t.lk(b));
      if (lead[b] == b) sg.off[u] = t.kv_off[b];
    }
  __syncthreads();
  // counts -> exclusive prefix (first[u + 1] holds group u's count)
  int32_t running = 0;
  for (int32_t c0 = 0; c0 < ngroups; c0 += kSchedThreads) {
    const int32_t u = c0 + tid;
    const int32_t incl = running + block_inclusive_scan_i32(u < ngroups ? sg.first[u + 1] : 0, s.wave_sums);
    if (u < ngroups) sg.first[u + 1] = incl;
    if (tid == kSchedThreads - 1) gs.carry = incl;
    __syncthreads();
    running = gs.carry;
  }
  __syncthreads();
  // d. a group's tasks in the order (prefix length, task): the order its work items walk them in, the same in every run
  for (int32_t b = tid; b < num_tasks; b += kSchedThreads)
    if (lead[b] >= 0) {
      const int32_t l = lead[b], lk = t.lk(b);
      int32_t before = 0;
      for (int32_t o = l; o < num_tasks; ++o)
        if (o != b && lead[o] == l) {
          const int32_t lko = t.lk(o);
          before += lko < lk || (lko == lk && o < b);
        }
      sg.tasks[sg.first[gid[l]] + before] = b;
    }
  // e. Groups must not overlap (tasks that share rows start at the same row); those that do are counted in word 3, from the stored rows
  // no group covers: before the first group, and from the end of a group to the start of the next.  (They stay in the table for whoever
  // reads a list back; fill_rows, in the launch's other workgroups, does not wait for it.)
  for (int32_t u = tid; u <= num_tasks; u += kSchedThreads) {
    int32_t lo = 0, hi = 0;
    if (u <= ngroups) {
      lo = u < ngroups ? sg.off[u] + sg.lmax[u] : 0;
      const int32_t from = u < ngroups ? sg.off[u] : -1;
      hi = total_k;
      for (int32_t o = 0; o < ngroups; ++o)
        if (sg.off[o] > from && sg.off[o] < hi) hi = sg.off[o];
      if (hi < lo) atomicAdd(&gs.violations, 1);
    }
    out.gap_lo[u] = lo;
    out.gap_hi[u] = hi;
  }
  __syncthreads();
  if (fits)
    for (int32_t u = tid; u <= num_tasks; u += kSchedThreads) {
      out.first[u] = sg.first[u];
      if (u < num_tasks) out.tasks[u] = sg.tasks[u], out.off[u] = sg.off[u], out.lmax[u] = sg.lmax[u];
    }
  const GroupUnits u{t, j.geom, sg.first, sg.tasks, sg.lmax};
  build_list<true>(s, u, ngroups, num_tasks, j.geom, j.ws, (int32_t)j.max_items, j.split);
  if (tid == 0) j.ws[3] = gs.violations;
}

// Zeroes the dk / dv rows that no work item writes.  Every workgroup finds the ranges of such rows and clears its share of each.
// Tasks that own their rows: those of tasks without queries, and the rows past the last task.  Tasks over shared rows: what lies
// between the ends of the stored documents that are read (for the longest task at every first row: up to the next first row), and before
// the first.
struct FillScratch {
  int32_t lo[kLdsTasks + 1], hi[kLdsTasks + 1], n;
};
__device__ void fill_rows(FillScratch &f, TaskCache &cache, const BwdFill &a, const ListJob &j, const int32_t *kv_off, int32_t num_tasks, int part, int parts) {
  const Tasks t = load_tasks(cache, j.cu_q, j.cu_k, kv_off, num_tasks);
  const int tid = threadIdx.x;
  for (int32_t b0 = 0; b0 <= num_tasks; b0 += kSchedThreads) {   // task `num_tasks` stands for the rows at the end (own) or at the start (shared)
    if (tid == 0) f.n = 0;
    __syncthreads();
    const int32_t b = b0 + tid;
    if (b <= num_tasks) {
      int32_t lo = 0, hi = 0;
      if (!kv_off) {
        if (b == num_tasks) lo = t.cu_k[num_tasks], hi = a.total_k;
        else if (t.lq(b) <= 0) lo = t.cu_k[b], hi = t.cu_k[b + 1];
      } else {
        auto live = [&](int32_t o) { return t.lq(o) > 0 && t.lk(o) > 0; };
        const bool start = b == num_tasks;
        if (start || live(b)) {
          const int32_t off = start ? -1 : t.kv_off[b], lk = start ? 0 : t.lk(b);
          lo = start ? 0 : off + lk;
          hi = a.total_k;
          for (int32_t o = 0; o < num_tasks; ++o) {
            if (!live(o)) continue;
            const int32_t oo = t.kv_off[o];
            if (oo == off && (t.lk(o) > lk || (t.lk(o) == lk && o < b))) lo = a.total_k;   // not the longest task of its document
            if (oo > off && oo < hi) hi = oo;
          }
        }
      }
      if (lo < 0) lo = 0;
      if (hi > a.total_k) hi = a.total_k;
      if (lo < hi) {
        const int32_t at = atomicAdd(&f.n, 1);
        f.lo[at] = lo;
        f.hi[at] = hi;
      }
    }
    __syncthreads();
    const int32_t rv = (int32_t)(a.row_bytes >> 4);   // vectors per row
    for (int32_t r = 0; r < f.n; ++r) {
      const int64_t v1 = (int64_t)f.hi[r] * rv;
      for (int64_t v = (int64_t)f.lo[r] * rv + (int64_t)part * kSchedThreads + tid; v < v1; v += (int64_t)parts * kSchedThreads) {
        if (a.shards.num_shards > 0) {
          const int32_t row = (int32_t)(v / rv);
          const int sh = find_shard(a.shards.row_start, a.shards.num_shards, row);
          const int64_t in_shard = (int64_t)(row - a.shards.row_start[sh]) * a.row_bytes + (v - (int64_t)row * rv) * 16;
          *reinterpret_cast<u32x4 *>(a.dk + a.shards.dk_off[sh] + in_shard) = u32x4{0, 0, 0, 0};
          *reinterpret_cast<u32x4 *>(a.dv + a.shards.dv_off[sh] + in_shard) = u32x4{0, 0, 0, 0};
        } else {
          reinterpret_cast<u32x4 *>(a.dk)[v] = u32x4{0, 0, 0, 0};
          reinterpret_cast<u32x4 *>(a.dv)[v] = u32x4{0, 0, 0, 0};
        }
      }
    }
    __syncthreads();
  }
}

// The row statistics, four lanes to a row, whose products are added up by the dQ kernel's instructions in its order: the same bits whichever makes them.
// Bound by reading dO and O, and by one trip to memory where those are few.
constexpr int kStatsRows = kSchedThreads / 4;
__device__ void row_stats(const RowStats &a, const int32_t *__restrict__ cu_q, int32_t num_tasks, int part, int parts) {
  const int quarter = threadIdx.x & 3;
  const int32_t rows = a.total_q * a.hq;
  for (int32_t r = part * kStatsRows + (int32_t)(threadIdx.x >> 2); r < rows; r += parts * kStatsRows) {
    const int32_t t = r / a.hq, h = r - t * a.hq;
    int64_t at = (int64_t)t * a.tok_bytes;
    if (a.task_off) {
      int32_t lo = 0, hi = num_tasks;   // the last task that starts at or before t
      while (hi - lo > 1) {
        const int32_t mid = (lo + hi) >> 1;
        if (cu_q[mid] <= t) lo = mid;
        else hi = mid;
      }
      if (t < cu_q[lo] || t >= cu_q[lo + 1]) continue;   // (no task's token)
      at = a.task_off[lo] + (int64_t)(t - cu_q[lo]) * a.tok_bytes;
    }
    const u32x4 *dop = reinterpret_cast<const u32x4 *>(a.dout + at + h * (kHeadDim * 2)) + quarter, *op = reinterpret_cast<const u32x4 *>(a.out + at + h * (kHeadDim * 2)) + quarter;
    u32x4 x[4], y[4];   // d = 32 s + 8 quarter .. +7
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = dop[4 * s], y[s] = op[4 * s];
    float lse = 0.f, sum = 0.f;
    if (quarter == 0) lse = a.lse ? a.lse[(int64_t)h * a.total_q + t] : reinterpret_cast<const float *>(a.lse_tok + at)[h];
#pragma unroll
    for (int s = 0; s < 4; ++s) sum = a.f16 ? add_products<true>(x[s], y[s], s, sum) : add_products<false>(x[s], y[s], s, sum);
    sum += __shfl_xor(sum, 1, 4);
    sum += __shfl_xor(sum, 2, 4);
    if (quarter == 0) {
      a.lse2[(int64_t)h * a.total_q + t] = lse * 1.4426950408889634f;
      a.neg_delta[(int64_t)h * a.total_q + t] = -sum;
    }
  }
}

// All that a backward needs before its kernels, in one launch: workgroup 0 builds the dK/dV list, workgroup 1 the dQ list, `fill_parts` others
// clear the dk / dv rows that no work item writes, and the rest makes the row statistics, where it is asked to.  (As launches of their own the three took 25 to 45 us of a small batch's backward.)
__global__ __launch_bounds__(kSchedThreads) void build_backward_kernel(ListJob kv, ListJob q, const int32_t *__restrict__ kv_off, int32_t num_tasks, BwdFill fill, int fill_parts, RowStats stats) {
  __shared__ TaskCache cache;
  __shared__ ListScratch s;
  __shared__ union {
    GroupScratch groups;
    FillScratch fill;
  } o;
  if (blockIdx.x == 0) {
    if (kv_off) build_shared(s, cache, o.groups, kv, kv_off, num_tasks, fill.total_k);
    else build_own<true>(s, cache, kv, num_tasks);
  } else if (blockIdx.x == 1) {
    build_own<false>(s, cache, q, num_tasks);
  } else if ((int)blockIdx.x < 2 + fill_parts) {
    fill_rows(o.fill, cache, fill, q, kv_off, num_tasks, (int)blockIdx.x - 2, fill_parts);
  } else {
    row_stats(stats, q.cu_q, num_tasks, (int)blockIdx.x - 2 - fill_parts, (int)gridDim.x - 2 - fill_parts);
  }
}

}  // namespace

int launch_build_forward(const ListJob &j, int32_t num_tasks, hipStream_t stream) {
  if (j.max_items > 0x7fffffff) return fail(DISTCA_E_INVALID, "schedule: too many work items");
  hipLaunchKernelGGL(build_forward_kernel, dim3(1), dim3(kSchedThreads), 0, stream, j, num_tasks);
  return check_launch("build_forward");
}

int launch_build_backward(const ListJob &kv, const ListJob &q, const int32_t *kv_off, int32_t num_tasks, const BwdFill &fill, const RowStats &stats, hipStream_t stream) {
  if (kv.max_items > 0x7fffffff || q.max_items > 0x7fffffff) return fail(DISTCA_E_INVALID, "schedule: too many work items");
  // (rows to clear are rare: a workgroup per MB of dk and dv, should it be all of them)
  const int64_t mb = (int64_t)fill.total_k * fill.row_bytes >> 19, parts = mb < 14 ? 14 : (mb > 254 ? 254 : mb);
  int64_t stat_parts = 0;
  if (stats.lse2) {
    stat_parts = ((int64_t)stats.total_q * stats.hq + kStatsRows - 1) / kStatsRows;
    if (stat_parts > 2 * num_compute_units()) stat_parts = 2 * num_compute_units();
  }
  hipLaunchKernelGGL(build_backward_kernel, dim3((unsigned)(2 + parts + stat_parts)), dim3(kSchedThreads), 0, stream, kv, q, kv_off, num_tasks, fill, (int)parts, stats);
  return check_launch("build_backward");
}

}  // namespace distca

using namespace distca;

namespace {
// The list of kind 0 (forward), 1 (dK/dV) or 2 (dQ) that a call with the preferred workspace launches over rows that tasks own.
struct LaunchedList {
  SchedGeom geom;
  int64_t max_blocks;
};
LaunchedList launched_list(int kind, const distca_ca_params *p) {
  const int64_t blocks = kind == 0 ? fwd_max_items(p) : dq_max_items(p);
  if (kind == 0) return {launched_fwd_geom(p, row_split_target(p, blocks, kCutFromTilesFwd)), blocks};
  if (kind == 1) return {launched_dkdv_geom(p, preferred_key_pieces(p), true, false, pair_backward(p, true)), bwd_key_blocks_own_rows(p)};
  return {launched_dq_geom(p, row_split_target(p, blocks, kCutFromTilesDq)), blocks};
}
}  // namespace

extern "C" int distca_ca_tile_shape(int kind, const distca_ca_params *p, int32_t out[2]) {
  if (!p || !out) return fail(DISTCA_E_INVALID, "tile_shape: null pointer");
  int rc = validate_params(p);
  if (rc) return rc;
  SchedGeom g = kind == 0 ? fwd_geom(p) : bwd_geom(p);
  out[0] = g.rows_per_block;  // flattened (token, head-in-group) rows
  out[1] = g.kv_per_block;
  return DISTCA_OK;
}

extern "C" int64_t distca_ca_schedule_capacity(int kind, const distca_ca_params *p) {
  if (!p) return fail(DISTCA_E_INVALID, "schedule_capacity: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  if (kind == 0) return fwd_max_items(p);
  if (kind == 1) return bwd_max_items(p);
  if (kind == 2) return dq_max_items(p);
  if (kind >= DISTCA_SCHED_LAUNCHED && kind <= DISTCA_SCHED_LAUNCHED + 2) {
    const LaunchedList l = launched_list(kind - DISTCA_SCHED_LAUNCHED, p);
    return l.max_blocks + l.geom.split_target;
  }
  return fail(DISTCA_E_INVALID, "schedule_capacity: kind must be 0 (fwd), 1 (bwd dK/dV) or 2 (bwd dQ), or one of these + %d", DISTCA_SCHED_LAUNCHED);
}

extern "C" int64_t distca_ca_schedule_host(int kind, const int32_t *cu_q, const int32_t *cu_k, const distca_ca_params *p,
                                           int32_t *items, int64_t max_items) {
  if (!p || !cu_q || !cu_k || (!items && max_items > 0)) return fail(DISTCA_E_INVALID, "schedule_host: null pointer");
  int rc = validate_params(p);
  if (rc) return rc;
  const bool launched = kind >= DISTCA_SCHED_LAUNCHED;
  if (kind != 0 && kind != 1 && !(launched && kind <= DISTCA_SCHED_LAUNCHED + 2))
    return fail(DISTCA_E_INVALID, "schedule_host: kind must be 0 (fwd) or 1 (bwd), or 0 to 2 + %d", DISTCA_SCHED_LAUNCHED);
  if (launched) kind -= DISTCA_SCHED_LAUNCHED;
  const LaunchedList list = launched ? launched_list(kind, p) : LaunchedList{kind == 0 ? fwd_geom(p) : bwd_geom(p), 0};
  const SchedGeom &g = list.geom;
  struct It { int32_t task, block, cost, bin, piece; };
  std::vector<It> whole, v;
  unsigned long long total_cost = 0;
  for (int32_t b = 0; b < p->num_tasks; ++b) {
    const int32_t lq = cu_q[b + 1] - cu_q[b], lk = cu_k[b + 1] - cu_k[b];
    const int32_t n = kind == 1 ? bwd_num_blocks(g, lq, lk) : fwd_num_items(g, lq, lk);
    for (int32_t i = 0; i < n; ++i) {
      const int32_t c = kind == 1 ? bwd_cost(g, lq, lk, i) : fwd_item_cost(g, lq, lk, i);
      whole.push_back({b, i, c, 0, 0});
      total_cost += (unsigned long long)c;
    }
  }
  int32_t piece = 0;
  if (g.split_target > 0) piece = piece_size(total_cost, g.split_target, g.min_piece);
  const bool fixed = g.units_per_head > 0;
  if (fixed) {
    std::vector<int32_t> bins;
    for (const It &w : whole) bins.push_back(cost_bin(g, w.cost));
    std::sort(bins.begin(), bins.end(), [](int32_t a, int32_t b) { return a > b; });
    int32_t ranked[4];
    for (int k = 0; k < 4; ++k) ranked[k] = (size_t)k * g.units_per_head < bins.size() ? bins[(size_t)k * g.units_per_head] << g.cost_shift : 0;
    piece = fixed_piece_size(g, total_cost, (int32_t)whole.size(), ranked, piece);
  }
  int64_t cut = 0, slots = 0;
  for (const It &w : whole) {
    const int32_t k = fixed ? fixed_piece_count(w.cost, piece) : piece_count(w.cost, piece);
    if (k > 1) ++cut, slots += k;
    for (int32_t j = 0; j < k; ++j) {
      int32_t lo, hi;
      piece_range(w.cost, j, k, fixed ? piece : 0, &lo, &hi);
      v.push_back({w.task, w.block, hi - lo, cost_bin(g, hi - lo), j | (k << 16)});
    }
  }
  if (launched && (cut > split_max_cut(list.max_blocks, g.split_target) || slots > split_max_slots(list.max_blocks, g.split_target)))
    return fail(DISTCA_E_WORKSPACE, "schedule_host: %lld blocks cut into %lld pieces, room for %lld into %lld", (long long)cut, (long long)slots,
                (long long)split_max_cut(list.max_blocks, g.split_target), (long long)split_max_slots(list.max_blocks, g.split_target));
  std::stable_sort(v.begin(), v.end(), [](const It &a, const It &b) { return a.bin > b.bin; });
  const int64_t n = (int64_t)v.size();
  if (kind == 1 && g.walk_round > 0)
    for (int64_t s0 = 0, s1; s0 < n; s0 = s1) {  // one cost bin: entries [s0, s1)
      for (s1 = s0 + 1; s1 < n && v[s1].bin == v[s0].bin; ++s1) {}
      for (int64_t e = s0; e < s1; ++e)
        if (((s1 - s0 <= kWalkTieLimit ? e : s0) / g.walk_round) & 1) v[e].piece |= kWalkUp;
    }
  for (int64_t e = 0; e < n && e < max_items; ++e) {
    items[4 * e + 0] = v[e].task;
    items[4 * e + 1] = v[e].block;
    items[4 * e + 2] = v[e].cost;
    items[4 * e + 3] = v[e].piece;
  }
  return n;
}
