// Varlen causal flash-attention forward for gfx950 (wave64, MFMA 16x16x32).
//
// Stands where the reference calls flash-attn's varlen forward
// (distca/runtime/megatron/ops/fused_comm_attn.py:151-197).
//
// Work decomposition.  The G = Hq/Hkv query heads that share a kv head are flattened with
// the tokens into one row axis: row R of a task = (token R / G, head R % G), so one K/V
// tile in LDS serves all heads of its group.  A workgroup (8 waves) owns kRows consecutive
// flattened rows of one task and one kv head and streams that task's visible KV prefix in
// tiles of 64 keys; tiles entirely above the diagonal are never visited and only tiles
// that straddle it are masked.  With 8 waves a workgroup covers 256 rows per K/V tile it pulls
// through the vector memory unit, whose throughput (about 64 bytes per clock per compute unit)
// is what a 128-row workgroup ran into.
//
// Per wave: 32 rows, two sub-blocks of 16, so that every K or V fragment read from LDS feeds two MFMAs.  Scores are produced transposed,
// S^T = K Q^T, so a lane holds one query row of each sub-block (column lane%16) and 4 keys per 16x16 block: the online-softmax
// row reductions are in-register plus an exchange among four lanes, and the fp32 accumulator
// registers of two blocks are, after conversion, already laid out as the B operand of
// O^T += V^T P^T.  Q stays in registers for the whole KV loop; K is read from LDS row-major
// (16-byte reads), V through the transposing LDS read.
//
// 16x16x32 MFMAs rather than 32x32x16: long prefixes are bound by power, and a FLOP of theirs moves half the accumulator bytes.  They leave fewer issue
// slots beside them (two vector instructions each, for five beside the larger one), and the softmax of a SIMD's other wave, some 120 vector instructions per 64
// MFMAs, does not fit: 131072 packed tokens went from 83 % of the pipe's cycles at 1.47 GHz to 70 % at 1.75.  us before -> after: those at 32/8 heads
// 12 150 -> 11 640, 8192 tokens 264 -> 254, a tick of 16384 tokens 1 339 -> 1 285, a lightly loaded server 261 -> 253, three documents (4096 tokens) 69.4 -> 68.8.  (Operands six steps ahead instead of four: 1 % slower; either half's waves at a higher
// priority: 1 to 2 % slower.)
//
// K/V tiles go from global memory straight into LDS (LDS-direct loads, four 256-byte rows per
// instruction, rows unpadded with swizzled 16-byte chunks, see tile_swz16), one period ahead of
// their use.
#include <type_traits>
#include <mutex>

#include "api_util.h"
#include "attn_bwd.h"
#include "attn_cfg.h"
#include "common.h"
#include "cut_blocks.h"
#include "kv_shards.h"

namespace distca {
namespace {

constexpr int kRowB = 256;    // bytes per K or V row in LDS (unpadded; chunk c of row r sits at c ^ tile_swz16(r))
constexpr int kKTile = kFwdKV * kRowB;
constexpr int kVTile = kFwdKV * kRowB;
constexpr int kKOff = 0, kVOff = 2 * kKTile;  // two K stages, then two V stages
// Behind the tiles the rows of Q on their way in, 8 KB of a wave's own, and half rows of O on their way out, 4 KB (see the epilogue); at 256
// registers a wave the workgroup has its compute unit, and its LDS, to itself anyway.
constexpr int kQOff = 2 * kKTile + 2 * kVTile, kQWave = 32 * kRowB;
constexpr int kOutOff = kQOff + kFwdWaves * kQWave, kOutWave = 32 * kRowB / 2;
constexpr int kFwdLds = kOutOff + kFwdWaves * kOutWave;
static_assert(kFwdLds <= 160 * 1024, "LDS of a compute unit");
constexpr int kDirectTasks = 256;    // batches without a list: at most so many tasks to look through
constexpr int kRankTasks = 64;       // ... or to find the block of a rank among
constexpr int kOutStores = 2 * 32 / 8;   // store instructions of a wave's rows
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// The wait in the form that the compiler takes into account: it then knows that Q is there (by its own count it would wait for it
// before every S, and with it for the tiles requested meanwhile).
template <int N>
__device__ __forceinline__ void wait_vm_known() {
  static_assert(N < 16, "the low four bits of the count");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | N);  // vmcnt(N), nothing of the other counters
  asm volatile("" ::: "memory");
}

// The MFMAs as assembly, their sums in place: of the builtin's, whose result need not be where C was, the compiler moves the accumulators round the
// registers and spaces LDS reads from MFMAs that still read what they overwrite.  It does not
// space these from the vector instructions that read their results: settle() does.
__device__ __forceinline__ void mfma16_in(f32x4 &acc, elemx8 a, elemx8 b) {  // acc += A B
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_in0(f32x4 &acc, elemx8 a, elemx8 b) {  // acc = A B
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
}
// What reads these sums stands behind it, eight wait states and more after the MFMA that made them.
__device__ __forceinline__ void settle(f32x4 (&x)[4][2]) {
  asm volatile("s_nop 7" : "+v"(x[0][0]), "+v"(x[0][1]), "+v"(x[1][0]), "+v"(x[1][1]), "+v"(x[2][0]), "+v"(x[2][1]), "+v"(x[3][0]), "+v"(x[3][1]));
}

struct FwdArgs {
  const elem_t *q, *k, *v;
  elem_t *out;
  float *lse;
  const int32_t *cu_q, *cu_k, *kv_off;
  const int32_t *sched;  // schedule workspace; null (SPLIT kernels): there is no list, num_tasks tasks' blocks are taken by rank, or, max_tiles == 0, as they come
  int32_t num_tasks, max_tiles;   // max_tiles: KV tiles of the longest prefix, at most
  const void *zero_row;  // 256 zero bytes: source of tile rows past the end of the prefix
  int32_t sched_items_off;  // int32 offset of the item array
  int32_t hq, hkv, group, total_q;
  int32_t causal;
  float scale;
  uint32_t group_magic;  // as in BwdArgs
  // Where the query and output tokens live.  Token t of task b starts at base + off[b] + t * tok_bytes
  // (off == nullptr: the packed tensor, off[b] = cu_q[b] * tok_bytes); head h at + h * 256 bytes.
  int32_t *tickets;  // one counter per kv head (sched.h)
  const int64_t *q_task_off, *out_task_off;
  int64_t q_tok_bytes, out_tok_bytes;
  int32_t merge_tiles;   // merged items: the list's merge_tiles (sched.h)
  int32_t lse_in_token;  // 1: lse of (token, head) as fp32 at token + hq * 256 + h * 4 (the [out | lse] reply), 0: lse[h][token]
  KvShards shards;       // SEG kernels: k and v are the bases of a buffer that holds the stored rows shard by shard
  const int32_t *cut, *slot;  // SPLIT kernels: the tables of a list with cut blocks (sched.h, SplitTables)
  uint8_t *partial;           // and the slots
};

// A piece's slot: O before normalisation as the accumulators lie, 16 bytes of a lane beside those of the next (a store of 1 KB
// per instruction), then (m, l) per row.
constexpr int64_t kFwdSlotStats = (int64_t)kFwdRows * kHeadDim * 4;
constexpr int64_t kFwdSlotBytes = kFwdSlotStats + kFwdRows * 8;

// Where lse of (token, head) goes, and, in the [out | lse] reply, the zeros behind the last head's.
__device__ __forceinline__ void store_lse(const FwdArgs &a, uint8_t *otok, int head, int64_t row, float lse) {
  if (a.lse_in_token) {
    float *lp = reinterpret_cast<float *>(otok + (int64_t)a.hq * kHeadDim * 2);
    lp[head] = lse;
    if (head == a.hq - 1) {  // zero the padding that rounds the token up to 16 bytes
      for (int64_t b = (int64_t)a.hq * (kHeadDim * 2 + 4); b < (((int64_t)a.hq * (kHeadDim * 2 + 4) + 15) & ~(int64_t)15); b += 4) *reinterpret_cast<float *>(otok + b) = 0.f;
    }
  } else {
    a.lse[(int64_t)head * a.total_q + row] = lse;
  }
}

__device__ __align__(256) unsigned char zero_row_static[256];   // the zero row of a call without a list; nothing writes it

// Block `e` of the batch's blocks of query rows, counted task after task, as a list's item: (task, block, -, one piece); task -1: none.
// Every wave finds it by a scan over 64 tasks at a time.
__device__ __forceinline__ int4 block_of_batch(const int32_t *cu_q, int num_tasks, int group, int e) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int b0 = 0; b0 < num_tasks; b0 += 64) {
    const int b = b0 + lane;
    const int lq = b < num_tasks ? cu_q[b + 1] - cu_q[b] : 0;
    const int n = lq > 0 ? (lq * group + kFwdRows - 1) / kFwdRows : 0;
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    const unsigned long long past = __ballot(before + incl > e);
    if (past) {
      const int l = __builtin_ctzll(past);
      return make_int4(b0 + l, e - before - __shfl(incl - n, l, 64), 0, 1 << 16);
    }
    before += __shfl(incl, 63, 64);
  }
  return make_int4(-1, 0, 0, 0);
}

// The block of rank `e` among the batch's blocks of query rows, from the one of the most KV tiles down.  Every wave finds it by itself, a lane to a
// task: a task's blocks cost the more the later they come, so that how many cost at least c is a division, and the cost at rank e a search over c, a
// sum over the lanes a step.
__device__ __forceinline__ int4 block_of_rank(const int32_t *cu_q, const int32_t *cu_k, int num_tasks, int group, int causal, int max_tiles, int e) {
  const int lane = threadIdx.x & 63;
  int lq = 0, lk = 0;
  if (lane < num_tasks) {
    lq = cu_q[lane + 1] - cu_q[lane];
    lk = cu_k[lane + 1] - cu_k[lane];
  }
  const int blocks = lq > 0 ? (lq * group + kFwdRows - 1) / kFwdRows : 0;
  // the first block of the lane's task that costs c or more: whose last token sees key kFwdKV (c - 1)
  auto first_of = [&](int c) {
    const int key = kFwdKV * (c - 1);
    const int t = causal ? key + 1 - (lk - lq) : 0;   // tokens of the task up to the first that sees it
    const int first = t > 1 ? ((t - 1) * group) / kFwdRows : 0;
    return c <= 0 ? 0 : key >= lk || t > lq ? blocks : first;
  };
  auto count = [&](int c) { return __builtin_amdgcn_readlane(wave_inclusive_scan_i32(blocks - first_of(c)), 63); };   // blocks of cost c or more
  int lo = 0, hi = max_tiles + 1, past = 0;   // count(lo) > e >= count(hi) = past
  if (e >= count(0)) return make_int4(-1, 0, 0, 0);
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1, n = count(mid);
    if (n > e) lo = mid;
    else hi = mid, past = n;
  }
  // block e - past of those of that cost, task after task
  // (prefixes longer than they were said to be count as that long)
  const int first = first_of(lo), n = (lo < max_tiles ? first_of(lo + 1) : blocks) - first, incl = wave_inclusive_scan_i32(n);
  const int task = __builtin_ctzll(__ballot(incl > e - past));
  return make_int4(task, e - past + __builtin_amdgcn_readlane(first - (incl - n), task), 0, 1 << 16);
}

// Draws a workgroup's item and kv head; false where none is left.
template <bool SPLIT>
__device__ __forceinline__ bool take_fwd_item(const FwdArgs &a, int32_t *slot, int &item, int &kvh, int4 &it) {
  if (SPLIT && !a.sched) {
    // no list (see run_fwd_tokens): the workgroup's id is its block's rank, or counts the batch's blocks
    item = (int)(blockIdx.x / (unsigned)a.hkv);
    kvh = (int)(blockIdx.x - (unsigned)item * (unsigned)a.hkv);
    it = a.max_tiles ? block_of_rank(a.cu_q, a.cu_k, a.num_tasks, a.group, a.causal, a.max_tiles, item) : block_of_batch(a.cu_q, a.num_tasks, a.group, item);
    return it.x >= 0;
  }
  const int nitems = a.sched[0];
  if (!take_item<SPLIT>(a.tickets, nitems, a.hkv, slot, item, kvh)) return false;
  it = reinterpret_cast<const int4 *>(a.sched + a.sched_items_off)[item];
  return true;
}

// SPLIT kernels: a piece is what a whole block over the keys from its first tile on would be: what counts keys from the start of the prefix is
// moved by the tiles before it, and below nothing knows of it.  (Carrying the first tile into the loops cost 5 % of a block's time.)
__device__ __forceinline__ void cut_out_piece(const FwdArgs &a, const int4 &it, int &ntiles, int &ks, int &lk, int &shift) {
  const int w = uniform_int(it.w);
  int tile0, tile1;
  piece_range(ntiles, item_piece(w), item_pieces(w), a.cut ? uniform_int(a.cut[2]) : 0, &tile0, &tile1);
  ntiles = tile1 - tile0;
  ks += tile0 * kFwdKV;
  lk -= tile0 * kFwdKV;
  shift -= tile0 * kFwdKV;
}

// SEG: K/V rows are addressed through a table of shards (kv_shards.h) instead of as one dense tensor.
// SPLIT (batches of few blocks): a work item may be a piece of a block, a range of its KV tiles (sched.h, piece_count), whose result
// goes to a slot; items are taken by workgroup id.
template <bool SEG, bool SPLIT>
__global__ __launch_bounds__(kFwdWaves * 64, 1) void ca_fwd_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  int item, kvh;
  int4 it;
  if (!take_fwd_item<SPLIT>(a, reinterpret_cast<int32_t *>(lds), item, kvh, it)) return;
  // (the item's fields and the task's bounds are moved to scalar registers as they are read: what derives from them,
  // base pointers, loop limits and tile addresses, is then scalar arithmetic)
  it.x = uniform_int(it.x);
  it.y = uniform_int(it.y);
  const int task = it.x;

  const int q0 = uniform_int(a.cu_q[task]);
  const int lq = uniform_int(a.cu_q[task + 1]) - q0;
  int lk = uniform_int(a.cu_k[task + 1]) - uniform_int(a.cu_k[task]);
  int ks = uniform_int(a.kv_off ? a.kv_off[task] : a.cu_k[task]);
  const int G = a.group;
  int shift = lk - lq;

  constexpr int kRows = kFwdRows;
  const int nrows = lq * G;
  const int mblk = it.y;
  elemx8 qf[2][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, c16 = lane & 15, g4 = lane >> 4;
  const int row_wg = mblk * kRows;
  auto div_group = [&](int n) { return a.group_magic ? (int)__umulhi((uint32_t)n, a.group_magic) : n; };

  // ---- KV extent of this workgroup
  int tok_end = (row_wg + kRows + G - 1) / G;
  if (tok_end > lq) tok_end = lq;
  int nvis = a.causal ? tok_end + shift : lk;
  if (nvis > lk) nvis = lk;
  int ntiles = nvis > 0 ? (nvis + kFwdKV - 1) / kFwdKV : 0;
  if constexpr (SPLIT) cut_out_piece(a, it, ntiles, ks, lk, shift);

  // ---- per-lane rows: row l32 of the wave where the results are stored, rows c16 and 16 + c16 in the MFMAs' operands and accumulators
  const uint8_t *qbytes = reinterpret_cast<const uint8_t *>(a.q) + uniform_int64(a.q_task_off ? a.q_task_off[task] : (int64_t)q0 * a.q_tok_bytes);
  uint8_t *obytes = reinterpret_cast<uint8_t *>(a.out) + uniform_int64(a.out_task_off ? a.out_task_off[task] : (int64_t)q0 * a.out_tok_bytes);
  int lim[2];   // the last key that the row sees
  {
    int lm = a.causal ? (row_wg + wave * 32 + l32) / G + shift : lk - 1;
    if (lm > lk - 1) lm = lk - 1;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) lim[rb] = __shfl(lm, 16 * rb + c16, 64);
  }
  // wave-uniform limits: first row's limit decides whether a tile needs masking, last row's
  // whether the wave has anything to do in it.
  const int wrow0 = row_wg + wave * 32;
  int wrow1 = wrow0 + 31;
  if (wrow1 > nrows - 1) wrow1 = nrows - 1;
  const bool wave_live = wrow0 < nrows;
  int lim_first = 0x7fffffff, lim_last = -1;
  if (wave_live) {
    lim_first = a.causal ? wrow0 / G + shift : lk - 1;
    if (lim_first > lk - 1) lim_first = lk - 1;
    lim_last = a.causal ? wrow1 / G + shift : lk - 1;
    if (lim_last > lk - 1) lim_last = lk - 1;
  }

  // ---- K/V tile fetch: wave w brings rows 16w .. 16w+15 of the K tile and of the V tile, four
  // rows per instruction; lane p fetches the chunk that belongs at chunk position p%16 of row p/16
  const int64_t kv_stride = (int64_t)a.hkv * kHeadDim;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(DISTCA_LDS uint8_t *)lds;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  // ---- Q: the wave's rows of the block whose first row is row0 come through LDS, four whole rows per instruction (a row past the task: the last
  // one again; nothing of it is stored), and each lane takes its fragments from there (B operand of S^T = K Q^T: row 16*rb + c16, d = 32*s + 8*g4 .. +7).
  // Loaded straight into that layout, an instruction touched 32 rows, and the address unit takes about a cycle for every line: of a 30 us block
  // of short documents these loads took one and a half.  us before -> after: documents of 128 to 2048 tokens (65536) 924 -> 881, three documents
  // (4096) 71.4 -> 69.8, 8192 tokens 270 -> 265, 389 tokens at 4/1 heads 15.7 -> 14.8, 131072 packed tokens 11 960 -> 11 920.
  auto request_q = [&](int row0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rl = 4 * i + (lane >> 4);
      int r = row0 + uwave * 32 + rl;
      if (r > nrows - 1) r = nrows - 1;
      const int t = div_group(r);
      const uint8_t *src = qbytes + (int64_t)t * a.q_tok_bytes + (kvh * G + (r - t * G)) * (kHeadDim * 2) + (((lane & 15) ^ tile_swz16(rl)) << 4);
      lds_direct_load16_ptr(src, lds0 + kQOff + uwave * kQWave + 4 * i * kRowB);
    }
  };
  auto take_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        qf[rb][s] = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(lds0 + kQOff + uwave * kQWave + (16 * rb + c16) * kRowB + (((4 * s + g4) ^ tile_swz16(c16)) << 4)));
  };
  request_q(row_wg);
  const elem_t *kbase = a.k + (SEG ? 0 : (int64_t)ks * kv_stride) + kvh * kHeadDim;
  const elem_t *vbase = a.v + (SEG ? 0 : (int64_t)ks * kv_stride) + kvh * kHeadDim;
  // SEG: the shards that hold the rows of the K tile and of the V tile requested next (the K requests run a tile ahead)
  ShardCursor kcur, vcur;
  if constexpr (SEG) {
    kcur.open(a.shards, SPLIT ? find_shard_wave(a.shards.row_start, a.shards.num_shards, ks) : a.shards.task_shard[task]);
    vcur = kcur;
  }
  // a wave brings kRowsW rows of a K tile or of a V tile, four rows per instruction
  constexpr int kRowsW = kFwdKV / kFwdWaves, kLdW = kRowsW / 4;
  auto issue_rows = [&](const elem_t *base, int j, uint32_t tile_off, const ShardCursor &cur, int which) {
#pragma unroll
    for (int i = 0; i < kLdW; ++i) {
      const int r = kRowsW * uwave + 4 * i + (lane >> 4);
      const int key = j * kFwdKV + r;
      const int chunk = (lane & 15) ^ tile_swz16(r);
      const elem_t *src;
      if constexpr (SEG) {
        src = reinterpret_cast<const elem_t *>(reinterpret_cast<const uint8_t *>(base) +
                                               (key < lk ? shard_row_offset(a.shards, cur, ks + key, which, kv_stride * 2) : 0));
      } else {
        src = base + (int64_t)key * kv_stride;
      }
      if (key >= lk) src = reinterpret_cast<const elem_t *>(SPLIT && !a.sched ? zero_row_static : a.zero_row);
      lds_direct_load16_ptr(src + chunk * 8, lds0 + tile_off + (kRowsW * uwave + 4 * i) * kRowB);
    }
  };
  // Tiles that lie wholly inside the prefix (all but the last one; SEG: and inside one shard) take a form without
  // per-lane address arithmetic: a scalar base that advances by one tile, plus a per-lane offset that never changes.
  uint32_t voff[kLdW];
#pragma unroll
  for (int i = 0; i < kLdW; ++i) {
    const int r = kRowsW * uwave + 4 * i + (lane >> 4);
    voff[i] = (uint32_t)((r * kv_stride + (((lane & 15) ^ tile_swz16(r)) * 8)) * 2);
  }
  auto issue_rows_fast = [&](const elem_t *tb, uint32_t tile_off) {
#pragma unroll
    for (int i = 0; i < kLdW; ++i) lds_direct_load16(tb, voff[i], lds0 + tile_off + (kRowsW * uwave + 4 * i) * kRowB);
  };
  // Key j * kFwdKV + r of a tile that ends at or before key `lim` lies at virt + (j * kFwdKV + r) * kv_stride.  Without
  // SEG that is the whole prefix but for its last, partial tile; with SEG the tiles inside the present shard: a tile
  // past `lim` looks for its shard (which moves virt and lim on) and only takes the per-lane form when it straddles
  // two shards or the end of the prefix, so that a run of tiles inside one shard costs what it costs without SEG.
  struct Run {
    const elem_t *virt;
    int lim;
  };
  Run krun{kbase, SEG ? 0 : lk}, vrun{vbase, SEG ? 0 : lk};
  auto issue_kv = [&](const elem_t *base, int j, uint32_t tile_off, Run &run, ShardCursor &cur, int which) __attribute__((always_inline)) {
    if ((j + 1) * kFwdKV <= run.lim) {
      issue_rows_fast(run.virt + (int64_t)j * kFwdKV * kv_stride, tile_off);
      return;
    }
    if constexpr (SEG) {
      const int r0 = ks + j * kFwdKV;
      cur.seek(a.shards, r0);
      if ((j + 1) * kFwdKV <= lk && cur.holds(r0, kFwdKV)) {
        run.virt = reinterpret_cast<const elem_t *>(static_cast<uintptr_t>(uniform_i64(
            (int64_t)reinterpret_cast<uintptr_t>(base) + (which ? cur.v : cur.k) - (int64_t)(cur.lo - ks) * kv_stride * 2)));
        run.lim = uniform_i32(cur.hi - ks < lk ? cur.hi - ks : lk);
        issue_rows_fast(run.virt + (int64_t)j * kFwdKV * kv_stride, tile_off);
        return;
      }
    }
    issue_rows(base, j, tile_off, cur, which);
  };
  auto issue_k = [&](int j) __attribute__((always_inline)) { issue_kv(kbase, j, kKOff + (j & 1) * kKTile, krun, kcur, 0); };
  auto issue_v = [&](int j) __attribute__((always_inline)) { issue_kv(vbase, j, kVOff + (j & 1) * kVTile, vrun, vcur, 1); };

  // ---- accumulators: a lane has column c16 of each, O^T: d = 16 db + 4 g4 + r, S^T: key 16 kb + 4 g4 + r
  f32x4 oacc[2][4][2];   // [db / 4][db % 4][rb]
  float m_run[2], mc_run[2], l_run[2];   // a row's reference, -c of it (infinity: there is none), and the lane's share of the sum
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
    for (int db = 0; db < 8; ++db) oacc[db >> 2][db & 3][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[rb] = -INFINITY;
    mc_run[rb] = INFINITY;
    l_run[rb] = 0.f;
  }
  const float c = a.scale * kLog2e;
  constexpr float kLazy = 8.f, kRedo = 32.f * 256.f;

  // LDS read offsets (bytes) that do not depend on the tile
  const int k_rd = c16 * kRowB + ((g4 ^ tile_swz16(c16)) << 4);  // + kb*16*kRowB, ^ 64*s
  // transposed V operand: lane points at (key 4 g4 + i4 [+ 16], chunk h1 [+ 2 db], half lane & 1)
  const int i4 = (lane & 15) >> 2, h1 = (lane & 3) >> 1;
  const int v_rd = (4 * g4 + i4) * kRowB + ((h1 ^ tile_swz16(4 * g4 + i4)) << 4) + 8 * (lane & 1);  // ^ 32*db

  // Absolute LDS addresses of this lane's operand reads in stage 0, the swizzled variants of each,
  // kept in registers: with the stage and the row block in the instruction's offset field, no address
  // arithmetic is left between the MFMAs.
  uint32_t k_ad[4], v_ad[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v_ad[i] = lds0 + kVOff + (v_rd ^ (i << 5));
    asm volatile("" : "+v"(v_ad[i]));
    if (i < 4) {
      k_ad[i] = lds0 + kKOff + (k_rd ^ (i << 6));
      asm volatile("" : "+v"(k_ad[i]));
    }
  }
  f32x4 sacc[4][2];
  elemx8 pf[2][2];
  auto tile_active = [&](int j) { return wave_live && j * kFwdKV <= lim_last; };
  auto nothing = [](auto...) {};
  using None = std::integral_constant<int, -1>;

  // ---- S^T = K Q^T : [64 keys] x [32 rows]
  constexpr int kPf = 4;  // K fragments are requested kPf steps, of two MFMAs each, before the MFMAs that use them
  elemx8 kf[kPf];
  auto load_k = [&](auto par, int f) __attribute__((always_inline)) {  // par: parity of the tile, known at compile time; f = 4*s + kb
    kf[f % kPf] = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(k_ad[f >> 2] + decltype(par)::value * kKTile + (f & 3) * 16 * kRowB));
  };
  auto first_k = [&](auto par) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < kPf; ++f) load_k(par, f);
  };
  // (the first fragments have been asked for; all_read() is called ahead of the last MFMAs, which need the last of them)
  auto phase_s = [&](auto par, auto all_read) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 16; ++f) {
      __builtin_amdgcn_sched_barrier(0);
      if (f == 14) all_read();
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        if (f < 4) mfma16_in0(sacc[f][rb], kf[f % kPf], qf[rb][0]);
        else mfma16_in(sacc[f & 3][rb], kf[f % kPf], qf[rb][f >> 2]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (f + kPf < 16) load_k(par, f + kPf);
    }
    settle(sacc);
  };
  // ---- mask, online softmax (log2 domain, a query row on four lanes), P as B operand
  auto phase_x = [&](int j, auto whole) __attribute__((always_inline)) {  // whole: every row of the wave sees the whole tile
    const int key0 = j * kFwdKV;
    if (!decltype(whole)::value && key0 + kFwdKV - 1 > lim_first) {  // the tile straddles the diagonal or the end of the prefix
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = key0 + 16 * kb + 4 * g4 + r;
            if (key > lim[rb]) sacc[kb][rb][r] = -INFINITY;
          }
    }
    // P = 2^(S c + mc) as B operand: slots 0 .. 3 of lane group g4 are keys 4 g4 .. +3 of a block of 16, slots 4 .. 7 those of the next; returns
    // this lane's share of the row sums
    auto exp_tile = [&](int rb, float mc) __attribute__((always_inline)) {
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          e[i] = fast_exp2(__builtin_fmaf(sacc[2 * t + (i >> 2)][rb][i & 3], c, mc));
          sum = t == 0 && i == 0 ? e[0] : sum + e[i];
        }
        pf[rb][t] = cvt8(e[0], e[1], e[2], e[3], e[4], e[5], e[6], e[7]);
      }
      return sum;
    };
    // The running reference m_run of a row need not be its maximum: any value within 2^kLazy of
    // it gives the same O / l.  So first try the tile against the old reference, without looking
    // for the maximum at all; only when a lane's 32 exponentials do not add up to at most 32 * 2^kLazy
    // (without a reference they add up to infinity or not at all) is the maximum taken, the rows rescaled if one moved by
    // more than 2^kLazy, and the tile done again.
    bool exact = !decltype(whole)::value && __any(m_run[0] == -INFINITY || m_run[1] == -INFINITY);
    float sum[2] = {0.f, 0.f};
    if (!exact) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) sum[rb] = exp_tile(rb, mc_run[rb]);
      exact = __any(!(sum[0] + sum[1] <= kRedo));
    }
    if (exact) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        float mx = sacc[0][rb][0];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = __builtin_fmaxf(mx, sacc[kb][rb][r]);
        mx = quad_max(mx);
        const float m_new = __builtin_fmaxf(m_run[rb], mx);
        if (__any((m_new - m_run[rb]) * c > kLazy)) {
          const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
          const float alpha = fast_exp2((m_run[rb] - m_use) * c);
          l_run[rb] *= alpha;
#pragma unroll
          for (int db = 0; db < 8; ++db)
#pragma unroll
            for (int r = 0; r < 4; ++r) oacc[db >> 2][db & 3][rb][r] *= alpha;
          m_run[rb] = m_new;
          mc_run[rb] = -m_new * c;
        }
        sum[rb] = exp_tile(rb, (m_run[rb] == -INFINITY) ? 0.f : mc_run[rb]);
      }
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) l_run[rb] += sum[rb];
  };
  // ---- O^T += V^T P^T : [128 d] x [32 rows], contraction over the 64 keys
  constexpr int kPfV = 4;  // V^T fragments are requested four steps, of two MFMAs each, ahead
  elemx4 vf[kPfV][2];
  auto load_v = [&](auto par, int u) __attribute__((always_inline)) {  // u = 8*t + db
    const uint32_t vo = decltype(par)::value * kVTile + 32 * (u >> 3) * kRowB;
    vf[u % kPfV][0] = lds_read_tr(lds_ptr(v_ad[u & 7] + vo));
    vf[u % kPfV][1] = lds_read_tr(lds_ptr(v_ad[u & 7] + vo + 16 * kRowB));
  };
  auto first_v = [&](auto par) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kPfV; ++u) load_v(par, u);
  };
  // (the first fragments have been asked for; next: the parity of the K tile whose first fragments to ask for, or None; beside(u) is
  // called after the MFMAs of step u)
  auto phase_pv = [&](auto par, auto next, auto beside) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) mfma16_in(oacc[(u >> 2) & 1][u & 3][rb], cat4(vf[u % kPfV][0], vf[u % kPfV][1]), pf[rb][u >> 3]);
      __builtin_amdgcn_sched_barrier(0);
      beside(u);
      if (u + kPfV < 16) load_v(par, u + kPfV);
      else if (decltype(next)::value >= 0 && u - (16 - kPfV) < kPf) load_k(next, u - (16 - kPfV));
    }
    if (decltype(next)::value < 0) {
      settle(oacc[0]);
      settle(oacc[1]);
    }
  };

  // The waves form two groups (0-3, 4-7; a SIMD holds one wave of each) that run half a period
  // apart, so that one group's MFMA phases coincide with the other's softmax arithmetic instead
  // of both queueing for the same pipe.  Between consecutive workgroup barriers b0, b1, b2, ...
  //   [b(2p),   b(2p+1)):  group 0: PV(p-1), S(p)     group 1: softmax(p-1)
  //   [b(2p+1), b(2p+2)):  group 0: softmax(p)        group 1: PV(p-1), S(p)
  // Tile p of K is read between b(2p) and b(2p+2), tile p of V between b(2p+2) and b(2p+4); every
  // wave requests K(p+1) and V(p) (those of period 0 ahead of the loop: below) after b(2p), into the stages whose last readers finished
  // before it, and waits for its own requests before b(2p+2).  The MFMA halves are the critical path of a period (one
  // group's, then the other's).  A request holds its wave for a hundred cycles or so: group 1 makes its requests right after b(2p), in
  // its softmax half; group 0 between MFMAs of PV(p-1) where it knows beforehand what to request (fast0), else behind b(2p+1) (in front
  // of its MFMA half they showed in the period, 3 %).
  // The first two K tiles and the first V tile are requested together ahead of the loop, so that a block waits for memory once: with
  // K(1) and V(0) requested in period 0, as the loop has it, that period (one tile's S to cover them) lasted as long as a second trip.
  // (Together with the rows of O leaving through LDS and Q known to be there, 131072 tokens in documents of 128 / 256 / 512 / 2048, 32/8
  // heads: 958 / 1010 / 1151 / 2798 -> 854 / 857 / 1014 / 2725 us; 131072 packed tokens 12.86 -> 12.72 ms.)
  auto request_first = [&](int n) __attribute__((always_inline)) {
    issue_k(0);
    issue_v(0);
    if (n > 1) issue_k(1);
  };
  const int grp = uwave >> 2;
  if (ntiles > 0) request_first(ntiles);
  wait_vm_known<0>();
  take_q();
  // the first period that makes requests of its own (opaque: known to the compiler, it becomes a first iteration of its own, and the
  // registers of the two spill)
  int requests_from = 1;
  asm volatile("" : "+s"(requests_from));
  __syncthreads();  // b0
  // The period loops are unrolled by two so that the LDS stage of every operand read is a constant folded into
  // the instruction's offset field instead of an addition per read between the MFMAs.
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // Between period 0 and fast_end the periods are of one kind for this wave: it sees the tile and the one before whole, and what they
  // request is whole and there, by scalar base.  They have loops of their own without conditions, in which S's first K fragments are asked for
  // beside the last MFMAs of PV, and b stands ahead of the last four MFMAs of S, when all reads of K are done.  With 32x32x16 MFMAs, us before -> after: 131072
  // packed tokens 13 240 -> 12 670, 8192 tokens 294 -> 282, a tick of 16384 tokens 1 483 -> 1 421, one over a document of 131072 29 390 ->
  // 27 930, forward of three documents (4096 tokens) 76.7 -> 74.7, lightly loaded server 276 -> 267; documents of 128 to 2048 tokens 980 -> 956.
  // (Of the 4.3 % the loops without conditions give 2.4, requests by a base that moves on 1.4, group 0's between MFMAs 0.5.  b ahead of the
  // softmax's last quarter, so that V's first fragments come meanwhile: 13 % slower; V's first fragments ahead of b in group 1: nothing;
  // K fragments three steps ahead: 2 % slower; group 0's requests three MFMAs earlier: 1.3 % slower.)
  int fast_end = wave_live ? (lim_first + 1) / kFwdKV : 0;
  if (fast_end > ntiles - 1) fast_end = ntiles - 1;
  if (!SEG && fast_end > lk / kFwdKV - 1) fast_end = lk / kFwdKV - 1;
  fast_end = uniform_int(fast_end);
  const int64_t tile_bytes = kFwdKV * kv_stride * 2;
  const uint8_t *k_next = reinterpret_cast<const uint8_t *>(kbase) + 2 * tile_bytes, *v_next = reinterpret_cast<const uint8_t *>(vbase) + tile_bytes;
  auto request_k = [&](auto par) __attribute__((always_inline)) {  // K(p + 1); par: parity of p
    issue_rows_fast(reinterpret_cast<const elem_t *>(k_next), kKOff + (1 - decltype(par)::value) * kKTile);
    k_next += tile_bytes;
  };
  auto request_v = [&](auto par) __attribute__((always_inline)) {  // V(p)
    issue_rows_fast(reinterpret_cast<const elem_t *>(v_next), kVOff + decltype(par)::value * kVTile);
    v_next += tile_bytes;
  };
  // (SEG: there is what lies inside the present shards)
  auto two_fast = [&](int p) __attribute__((always_inline)) {
    return p + 1 < fast_end && (!SEG || ((p + 3) * kFwdKV <= krun.lim && (p + 2) * kFwdKV <= vrun.lim));
  };
  auto enter_fast = [&](int p) __attribute__((always_inline)) {
    if constexpr (SEG) {
      k_next = reinterpret_cast<const uint8_t *>(krun.virt) + (p + 1) * tile_bytes;
      v_next = reinterpret_cast<const uint8_t *>(vrun.virt) + p * tile_bytes;
    }
  };
  auto fast0 = [&](int p, auto par) __attribute__((always_inline)) {
    using Same = std::integral_constant<int, decltype(par)::value>;
    using Other = std::integral_constant<int, 1 - decltype(par)::value>;
    first_v(Other{});
    phase_pv(Other{}, Same{}, [&](int u) __attribute__((always_inline)) {
      if (u == 4) request_k(par);
      if (u == 8) request_v(par);
    });
    phase_s(Same{}, barrier);
    phase_x(p, std::true_type{});
    wait_vm0();
    barrier();
  };
  auto fast1 = [&](int p, auto par) __attribute__((always_inline)) {
    using Same = std::integral_constant<int, decltype(par)::value>;
    using Other = std::integral_constant<int, 1 - decltype(par)::value>;
    request_k(par);
    request_v(par);
    phase_x(p - 1, std::true_type{});
    barrier();
    first_v(Other{});
    phase_pv(Other{}, Same{}, nothing);
    phase_s(Same{}, [&]() __attribute__((always_inline)) { wait_vm0(); barrier(); });
  };
  auto slow0 = [&](int p, auto par) __attribute__((always_inline)) {   // par = parity of p
    using Same = std::integral_constant<int, decltype(par)::value>;
    using Other = std::integral_constant<int, 1 - decltype(par)::value>;
    if (p > 0 && tile_active(p - 1)) { first_v(Other{}); phase_pv(Other{}, None{}, nothing); }
    const bool act = p < ntiles && tile_active(p);
    if (act) { first_k(Same{}); phase_s(Same{}, nothing); }
    __syncthreads();
    if (p >= requests_from) {
      if (p + 1 < ntiles) issue_k(p + 1);
      if (p < ntiles) issue_v(p);
    }
    if (act) phase_x(p, std::false_type{});
    if (p >= requests_from) wait_vm0();
    __syncthreads();
  };
  auto slow1 = [&](int p, auto par) __attribute__((always_inline)) {
    using Same = std::integral_constant<int, decltype(par)::value>;
    using Other = std::integral_constant<int, 1 - decltype(par)::value>;
    if (p >= requests_from) {
      if (p + 1 < ntiles) issue_k(p + 1);
      if (p < ntiles) issue_v(p);
    }
    const bool act_prev = p > 0 && tile_active(p - 1);
    if (act_prev) phase_x(p - 1, std::false_type{});
    __syncthreads();
    if (act_prev) { first_v(Other{}); phase_pv(Other{}, None{}, nothing); }
    if (p < ntiles && tile_active(p)) { first_k(Same{}); phase_s(Same{}, nothing); }
    if (p >= requests_from) wait_vm0();
    __syncthreads();
  };
  int p = 1;
  auto work_off = [&](auto fast, auto slow) __attribute__((always_inline)) {
    auto fast_periods = [&]() __attribute__((always_inline)) {
      for (enter_fast(p); two_fast(p); p += 2) {
        fast(p, P1{});
        fast(p + 1, P0{});
      }
    };
    if constexpr (SEG) {
      // Period 0 inside the loop, whose periods with conditions come back at every end of a shard: the compiler then makes less of them (a forward over 22 shards, a launch:
      // 6.33e8 -> 6.27e8 vector instructions, wave-cycles at a wait 6.5e8 -> 6.0e8 units of four; not the size of the code, 77 -> 64 KB: 7e3 and 4e3 misses in 2.2e8
      // requests).  us, in-place ticks with period 0 of its own / so: 8192 tokens of 8 ranks at 64/8 heads 3 343 / 3 288, one document 6 457 / 6 372, 4096 of 4 at 32/8
      // 147 / 144, 8192 of 8 at 32/8 1 584 / 1 558.
      p = -1;   // (opaque: known to the compiler, the first turn becomes one of its own)
      asm volatile("" : "+s"(p));
      for (; p <= ntiles; p += 2) {
        if (p > 0) {
          fast_periods();  // (the period below may have found the next shard)
          slow(p, P1{});
        }
        if (p + 1 <= ntiles) slow(p + 1, P0{});
      }
      return;
    }
    slow(0, P0{});
    fast_periods();
    for (; p <= ntiles; p += 2) {
      slow(p, P1{});
      if (p + 1 <= ntiles) slow(p + 1, P0{});
    }
  };
  if (grp == 0) work_off(fast0, slow0);
  else work_off(fast1, slow1);

  const int row = row_wg + wave * 32 + l32, tok = div_group(row);
  uint8_t *otok = obytes + (int64_t)tok * a.out_tok_bytes;

  if constexpr (SPLIT) {
    const int slot = a.slot ? uniform_int(a.slot[2 * item]) : -1;
    if (slot >= 0) {
      // d0 = 16 db + 4 g4 of row r of the wave at d block db % 4, quarter 2 (db / 4) + g4 / 2, lane 32 (g4 % 2) + r (cut_blocks.h)
      uint8_t *at = a.partial + ((int64_t)slot * a.hkv + kvh) * kFwdSlotBytes;
      f32x4 *op = reinterpret_cast<f32x4 *>(at) + wave * 16 * 64 + (g4 >> 1) * 64 + (g4 & 1) * 32 + c16;
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) op[(4 * (db & 3) + 2 * (db >> 2)) * 64 + 16 * rb] = oacc[db >> 2][db & 3][rb];
      const float l0 = quad_sum(l_run[0]), l1 = quad_sum(l_run[1]);
      if (lane < 32) reinterpret_cast<f32x2 *>(at + kFwdSlotStats)[wave * 32 + l32] = g4 ? f32x2{m_run[1], l1} : f32x2{m_run[0], l0};
      return;
    }
  }

  // ---- epilogue: normalise, write O and LSE (fp32, natural log).  A lane holds a quarter of its two rows in pieces of 8 bytes (block db
  // holds d = 16 db + 4 g4 .. +3); stored from there, an instruction touched 16 rows.  The pieces go to the wave's
  // 4 KB of LDS, half of every row at a time, and leave from there in whole
  // cache lines, eight rows per instruction.
  {
    float l_tot[2], inv[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      l_tot[rb] = quad_sum(l_run[rb]);
      inv[rb] = l_tot[rb] > 0.f ? 1.f / l_tot[rb] : 0.f;
    }
    const uint32_t out_w = lds0 + kOutOff + uwave * kOutWave;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // half rows: d = 64 h .. 64 h + 63
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int db = 4 * h; db < 4 * h + 4; ++db) {
          const int chunk = 2 * (db & 3) + (g4 >> 1);   // half g4 & 1 of it
          const f32x4 &o = oacc[h][db & 3][rb];
          *static_cast<DISTCA_LDS elemx4 *>(const_cast<DISTCA_LDS void *>(lds_ptr(out_w + (16 * rb + c16) * (kRowB / 2) + ((chunk ^ (c16 & 7)) << 4) + 8 * (g4 & 1)))) =
              cvt4(o[0] * inv[rb], o[1] * inv[rb], o[2] * inv[rb], o[3] * inv[rb]);
        }
      // (LDS operations of one wave complete in order: the reads below see the writes above, and the second half's writes come behind them)
#pragma unroll
      for (int i = 0; i < kOutStores / 2; ++i) {
        const int rl = 8 * i + (lane >> 3);
        const int r = row_wg + uwave * 32 + rl;
        const elemx8 o8 = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(out_w + rl * (kRowB / 2) + (((lane & 7) ^ (rl & 7)) << 4)));
        if (r < nrows) {
          const int t = div_group(r);
          *reinterpret_cast<elemx8 *>(reinterpret_cast<elem_t *>(obytes + (int64_t)t * a.out_tok_bytes) + (kvh * G + (r - t * G)) * kHeadDim + 64 * h + 8 * (lane & 7)) = o8;
        }
      }
    }
    if (row < nrows && lane < 32) {   // lane l32 has the sums of its row as those of row g4 of the two
      const int hg = row - tok * G;
      const float l = g4 ? l_tot[1] : l_tot[0], m = g4 ? m_run[1] : m_run[0];
      const float lse = l > 0.f ? (m * c + fast_log2(l)) * kLn2 : -INFINITY;
      store_lse(a, otok, kvh * G + hg, q0 + tok, lse);
    }
  }
}

#include "attn_fwd32.inc"

// Adds up the pieces of the blocks that were cut, in their order (cut_blocks.h; a workgroup has the rows of one wave, a lane what it held
// in the kernel above).  Bound by reading the slots (128 KB a piece), four pieces' loads in flight at a time.
__global__ __launch_bounds__(kCutThreads) void ca_fwd_combine_kernel(FwdArgs a) {
  static_assert(kFwdWaves == kCutParts, "a part is a wave's rows");
  const int kvh = blockIdx.y, wave = blockIdx.z, lane = threadIdx.x & 63, db = threadIdx.x >> 6, l32 = lane & 31, g = lane >> 5, G = a.group;
  const float c = a.scale * kLog2e;
  auto token_at = [&](const int4 &e, int r, int &tok, int &head) -> uint8_t * {  // of the output, null if there is no such row
    const int q0 = a.cu_q[e.x], nrows = (a.cu_q[e.x + 1] - q0) * G, row = e.y * kFwdRows + wave * 32 + r;
    tok = row / G;
    head = kvh * G + row - tok * G;
    uint8_t *at = reinterpret_cast<uint8_t *>(a.out) + (a.out_task_off ? a.out_task_off[e.x] : (int64_t)q0 * a.out_tok_bytes) + (int64_t)tok * a.out_tok_bytes;
    tok += q0;
    return row < nrows ? at : nullptr;
  };
  add_up_cut_blocks(
      a.cut, a.slot,
      [&](const int4 &e, f32x4 (&o)[4]) {
        const int pieces = e.z;
        const uint8_t *first = a.partial + ((int64_t)e.w * a.hkv + kvh) * kFwdSlotBytes;
        const int64_t step = a.hkv * kFwdSlotBytes;
        auto stat = [&](int j) { return reinterpret_cast<const f32x2 *>(first + j * step + kFwdSlotStats)[wave * 32 + l32]; };
        f32x4 v[4][4];
        f32x2 s[4];
        auto load = [&](int j) __attribute__((always_inline)) {  // pieces j .. j + 3, as far as there are
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (j + u < pieces) {
              s[u] = stat(j + u);
              const f32x4 *op = reinterpret_cast<const f32x4 *>(first + (j + u) * step) + (wave * 16 + 4 * db) * 64 + lane;
#pragma unroll
              for (int cq = 0; cq < 4; ++cq) v[u][cq] = op[cq * 64];
            }
        };
        load(0);
        float m = -INFINITY;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (u < pieces) m = __builtin_fmaxf(m, s[u][0]);
#pragma unroll 4
        for (int j = 4; j < pieces; ++j) m = __builtin_fmaxf(m, stat(j)[0]);
        float l = 0.f;
        for (int j = 0; j < pieces; j += 4) {
          if (j > 0) load(j);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (j + u < pieces) {
              const float w = s[u][0] == -INFINITY ? 0.f : fast_exp2((s[u][0] - m) * c);
              l += w * s[u][1];
#pragma unroll
              for (int cq = 0; cq < 4; ++cq)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[cq][r] = __builtin_fmaf(w, v[u][cq][r], o[cq][r]);
            }
        }
        const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
        for (int cq = 0; cq < 4; ++cq)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[cq][r] *= inv;
        if (db == 0 && g == 0) {
          int tok, head;
          if (uint8_t *otok = token_at(e, l32, tok, head)) store_lse(a, otok, head, tok, l > 0.f ? (m * c + fast_log2(l)) * kLn2 : -INFINITY);
        }
      },
      [&](const int4 &e, int r) -> elem_t * {
        int tok, head;
        uint8_t *otok = token_at(e, r, tok, head);
        return otok ? reinterpret_cast<elem_t *>(otok) + head * kHeadDim : nullptr;
      });
}

// How a forward is laid out in its workspace: the list, and, when blocks are cut, the tables and slots of the pieces.
struct FwdLayout {
  int64_t max_blocks, max_items, tables, slots, total;
  int32_t target;
};
FwdLayout fwd_layout(const distca_ca_params *p, bool split) {
  FwdLayout w;
  w.max_blocks = fwd_max_items(p);
  w.target = split ? row_split_target(p, w.max_blocks, kCutFromTilesFwd) : 0;
  w.max_items = w.max_blocks + w.target;
  w.tables = align_up(sched_region_bytes(p->num_tasks, w.max_items), 256);
  w.slots = w.tables + split_tables_bytes(w.max_blocks, w.target, w.max_items);
  w.total = w.target > 0 ? w.slots + split_max_slots(w.max_blocks, w.target) * p->num_heads_kv * kFwdSlotBytes : sched_region_bytes(p->num_tasks, w.max_items);
  return w;
}

}  // namespace
}  // namespace distca

using namespace distca;

#ifndef DISTCA_F16
// Scratch memory of distca_ca_fwd_noalloc: the forward's work list, zero row and ticket counters, which every other
// entry point takes from the caller's workspace.  One copy per GPU, held until the process ends.  The name below is
// a host-side stand-in, never a device address: host code uses the per-device address from hipGetSymbolAddress.
constexpr int64_t kNoAllocScratchBytes = 1 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
// Device address of `scratch` on the current device, resolved once per device with that device current.
int noalloc_scratch(void **out) {
  static std::mutex mu;
  static void *ptr[64] = {nullptr};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(DISTCA_E_LAUNCH, "ca_fwd_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= 64) return fail(DISTCA_E_UNSUPPORTED, "ca_fwd_noalloc: device id %d (at most 64 devices)", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(DISTCA_E_LAUNCH, "ca_fwd_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    ptr[dev] = p;
  }
  *out = ptr[dev];
  return DISTCA_OK;
}
}  // namespace

extern "C" int64_t distca_ca_fwd_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int64_t distca_ca_fwd_workspace_bytes(const distca_ca_params *p) {
  if (!p) return fail(DISTCA_E_INVALID, "fwd_workspace_bytes: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  return fwd_layout(p, false).total;
}
extern "C" int64_t distca_ca_fwd_workspace_preferred_bytes(const distca_ca_params *p) {
  if (!p) return fail(DISTCA_E_INVALID, "fwd_workspace_preferred_bytes: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  return fwd_layout(p, true).total;
}

extern "C" int distca_ca_fwd_tokens(const void *q_base, const int64_t *q_task_off, int64_t q_tok_bytes, const void *k,
                                    const void *v, void *out_base, const int64_t *out_task_off, int64_t out_tok_bytes,
                                    float *lse, const int32_t *cu_q, const int32_t *cu_k, const int32_t *kv_off,
                                    const distca_ca_params *p, void *workspace, int64_t workspace_bytes, void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_fwd: null params");
  return (p->dtype == DISTCA_DTYPE_F16 ? run_fwd_tokens_f16 : run_fwd_tokens)(q_base, q_task_off, q_tok_bytes, k, v, nullptr, out_base,
                                                                              out_task_off, out_tok_bytes, lse, cu_q, cu_k, kv_off, p,
                                                                              workspace, workspace_bytes, stream);
}

extern "C" int distca_ca_fwd_buffers(const void *q_base, const int64_t *q_task_off, int64_t q_tok_bytes, const void *k,
                                     const void *v, const distca_kv_shards *kv_shards, void *out_base, const int64_t *out_task_off,
                                     int64_t out_tok_bytes, float *lse, const int32_t *cu_q, const int32_t *cu_k,
                                     const int32_t *kv_off, const distca_ca_params *p, void *workspace, int64_t workspace_bytes,
                                     void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_fwd: null params");
  if (!kv_shards) return fail(DISTCA_E_INVALID, "ca_fwd_buffers: null table of K/V shards");
  return (p->dtype == DISTCA_DTYPE_F16 ? run_fwd_tokens_f16 : run_fwd_tokens)(q_base, q_task_off, q_tok_bytes, k, v, kv_shards, out_base,
                                                                              out_task_off, out_tok_bytes, lse, cu_q, cu_k, kv_off, p,
                                                                              workspace, workspace_bytes, stream);
}

namespace distca {
int make_kv_shards(const distca_kv_shards *in, const int32_t *kv_off, bool backward, KvShards *out) {
  if (in->num_shards <= 0) return fail(DISTCA_E_INVALID, "kv_shards: num_shards=%d", in->num_shards);
  if (!in->row_start || !in->k_offset || !in->v_offset || !in->task_shard) return fail(DISTCA_E_INVALID, "kv_shards: null array");
  if (backward && (!in->dk_offset || !in->dv_offset)) return fail(DISTCA_E_INVALID, "kv_shards: the backward needs dk_offset and dv_offset");
  if (!kv_off) return fail(DISTCA_E_INVALID, "kv_shards: kv_task_offsets is required (tasks name stored rows)");
  out->row_start = in->row_start; out->k_off = in->k_offset; out->v_off = in->v_offset;
  out->dk_off = in->dk_offset; out->dv_off = in->dv_offset; out->task_shard = in->task_shard;
  out->num_shards = in->num_shards;
  return DISTCA_OK;
}
}  // namespace distca

extern "C" int distca_ca_fwd(const void *q, const void *k, const void *v, void *out, float *lse, const int32_t *cu_q,
                             const int32_t *cu_k, const int32_t *kv_off, const distca_ca_params *p, void *workspace,
                             int64_t workspace_bytes, void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_fwd: null params");
  const int rc = validate_params(p);
  if (rc) return rc;
  if (p->num_tasks == 0 || p->total_q == 0) return DISTCA_OK;
  if (!lse) return fail(DISTCA_E_INVALID, "ca_fwd: null pointer");
  return distca_ca_fwd_tokens(q, nullptr, 0, k, v, out, nullptr, 0, lse, cu_q, cu_k, kv_off, p, workspace, workspace_bytes, stream);
}

extern "C" int distca_ca_fwd_noalloc(const void *q, const void *k, const void *v, void *out, float *lse, const int32_t *cu_q,
                                     const int32_t *cu_k, const int32_t *kv_off, const distca_ca_params *p, void *stream) {
  if (!p) return fail(DISTCA_E_INVALID, "ca_fwd_noalloc: null params");
  const int64_t need = distca_ca_fwd_workspace_bytes(p);
  if (need < 0) return (int)need;
  if (need > kNoAllocScratchBytes)
    return fail(DISTCA_E_WORKSPACE,
                "ca_fwd_noalloc: this batch needs %lld B of scratch, the static array holds %lld B (about %lld work items: "
                "query rows x heads per kv head / %d + tasks); use distca_ca_fwd with a workspace",
                (long long)need, (long long)kNoAllocScratchBytes, (long long)(kNoAllocScratchBytes / 16), kFwdRows);
  void *ws = nullptr;
  const int rc = noalloc_scratch(&ws);
  if (rc) return rc;
  return distca_ca_fwd(q, k, v, out, lse, cu_q, cu_k, kv_off, p, ws, need, stream);
}

#endif  // !DISTCA_F16

namespace distca {
int DISTCA_FN(run_fwd_tokens)(const void *q_base, const int64_t *q_task_off, int64_t q_tok_bytes, const void *k, const void *v,
                              const distca_kv_shards *kv_shards, void *out_base, const int64_t *out_task_off, int64_t out_tok_bytes,
                              float *lse, const int32_t *cu_q, const int32_t *cu_k, const int32_t *kv_off, const distca_ca_params *p,
                              void *workspace, int64_t workspace_bytes, void *stream) {
  const void *q = q_base;
  void *out = out_base;
  if (!p) return fail(DISTCA_E_INVALID, "ca_fwd: null params");
  int rc = validate_params(p);
  if (rc) return rc;
  if (p->num_tasks == 0 || p->total_q == 0) return DISTCA_OK;
  if (!q || !k || !v || !out || !cu_q || !cu_k) return fail(DISTCA_E_INVALID, "ca_fwd: null pointer");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return fail(DISTCA_E_INVALID, "ca_fwd: q/k/v/out must be 16-byte aligned");
  if (!lse && !out_task_off) return fail(DISTCA_E_INVALID, "ca_fwd: lse is null and the output is not in token layout");
  const int64_t row_bytes = (int64_t)p->num_heads_q * kHeadDim * 2;
  if (!q_task_off) q_tok_bytes = row_bytes;
  if (!out_task_off) out_tok_bytes = row_bytes;
  if (q_tok_bytes < row_bytes || (q_tok_bytes & 15)) return fail(DISTCA_E_INVALID, "ca_fwd: query token of %lld B (needs >= %lld, multiple of 16)", (long long)q_tok_bytes, (long long)row_bytes);
  const int64_t out_need = row_bytes + (lse ? 0 : (int64_t)p->num_heads_q * 4);
  if (out_tok_bytes < out_need || (out_tok_bytes & 15)) return fail(DISTCA_E_INVALID, "ca_fwd: output token of %lld B (needs >= %lld, multiple of 16)", (long long)out_tok_bytes, (long long)out_need);
  const int64_t need = distca_ca_fwd_workspace_bytes(p);
  if (!workspace || workspace_bytes < need) return fail(DISTCA_E_WORKSPACE, "ca_fwd: workspace %lld B < required %lld B", (long long)workspace_bytes, (long long)need);
  if (!aligned16(workspace)) return fail(DISTCA_E_INVALID, "ca_fwd: workspace must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  FwdLayout lay = fwd_layout(p, true);
  if (lay.target > 0 && workspace_bytes < lay.total) lay = fwd_layout(p, false);   // no room for pieces
  const int64_t max_items = lay.max_items;
  const bool split = lay.target > 0, few = few_row_blocks(p);
  const SchedGeom geom = launched_fwd_geom(p, lay.target);
  const SplitTables tables = split ? split_tables((uint8_t *)workspace + lay.tables, lay.max_blocks, lay.target) : SplitTables{};
  // A batch whose blocks all run at once (one workgroup a compute unit) and stay whole needs no list: which workgroup has which block
  // does not matter then, and finding one by a scan of the task bounds takes one trip to memory where the list takes a launch of 5 us.
  // us with a list / without: 256 tokens at 4/1 heads 17.3 / 12.4, 389 at 8/2 20.0 / 15.1, 1000 at 32/8 31.9 / 26.9.
  const bool at_once = max_items * p->num_heads_kv <= num_compute_units() && p->num_tasks <= kDirectTasks;
  // With several rounds of workgroups, which take their items by id here, the order matters, longest first; up to 64 tasks a workgroup finds the block of
  // its rank in less than a microsecond a round.  us with a list / without: 2048 tokens at 32/8 heads 50.2 / 45.3, 512 + 1024 + 2560 70.6 / 66.7, 4096 123.0 /
  // 118.8, 20 x 300 50.8 / 47.4, 16 x 1024 at 8/2 45.4 / 41.0, 6 blocks a unit (12000 at 32/8) 918 / 917.  (Four tasks a lane, up to 256: a microsecond
  // more a round, most of it for code that is not in the cache yet, and no gain left.)
  const bool direct = few && !split && (at_once || p->num_tasks <= kRankTasks);
  if (!direct) {
    rc = launch_build_forward(ListJob{cu_q, cu_k, geom, (int32_t *)workspace, max_items, tables}, p->num_tasks, s);
    if (rc) return rc;
  }

  FwdArgs a;
  a.q = (const elem_t *)q; a.k = (const elem_t *)k; a.v = (const elem_t *)v;
  a.out = (elem_t *)out; a.lse = lse;
  a.cu_q = cu_q; a.cu_k = cu_k; a.kv_off = kv_off;
  a.sched = direct ? nullptr : (const int32_t *)workspace;
  a.num_tasks = p->num_tasks;
  a.max_tiles = at_once ? 0 : p->max_seqlen_k / kFwdKV + 1;
  a.zero_row = (const uint8_t *)workspace + sched_zero_row_off(p->num_tasks, max_items);
  a.sched_items_off = (int32_t)sched_header_ints(p->num_tasks);
  a.tickets = (int32_t *)((uint8_t *)workspace + sched_ticket_off(p->num_tasks, max_items));
  a.hq = p->num_heads_q; a.hkv = p->num_heads_kv; a.group = p->num_heads_q / p->num_heads_kv;
  a.total_q = p->total_q; a.causal = p->causal != 0; a.scale = p->softmax_scale;
  a.group_magic = a.group == 1 ? 0u : (uint32_t)(((1ull << 32) + a.group - 1) / a.group);
  a.q_task_off = q_task_off; a.out_task_off = out_task_off; a.q_tok_bytes = q_tok_bytes; a.out_tok_bytes = out_tok_bytes;
  a.lse_in_token = lse ? 0 : 1;
  a.merge_tiles = geom.merge_tiles;
  a.cut = tables.cut; a.slot = tables.slot; a.partial = (uint8_t *)workspace + lay.slots;
  a.shards = KvShards{};
  if (kv_shards) {
    rc = make_kv_shards(kv_shards, kv_off, false, &a.shards);
    if (rc) return rc;
  }
  const int64_t grid = list_grid(p, max_items, few);
  if (grid > 0x7fffffff) return fail(DISTCA_E_INVALID, "ca_fwd: grid too large");
  if (device_setup_pending(kSlotFwdLds)) {
    const void *kernels[] = {(const void *)ca_fwd_kernel<false, false>, (const void *)ca_fwd_kernel<true, false>,
                             (const void *)ca_fwd_kernel<false, true>,    (const void *)ca_fwd_kernel<true, true>,
                             (const void *)ca_fwd32_kernel<false, true>,  (const void *)ca_fwd32_kernel<true, true>,
                             (const void *)ca_fwd32_kernel<false, false>, (const void *)ca_fwd32_kernel<true, false>};
    for (const void *kf : kernels) {
      hipError_t e = hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, kFwdLds);
      if (e != hipSuccess) return fail(DISTCA_E_LAUNCH, "ca_fwd: cannot reserve %d B of LDS: %s", kFwdLds, hipGetErrorString(e));
    }
    device_setup_done(kSlotFwdLds);
  }
  {
    ScopedTimer timer(DISTCA_TIMER_CA_FWD, s);
    const dim3 g((unsigned)grid), b(kFwdWaves * 64);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, kFwdLds, s, a); };
    if (few && fwd_mfma32(p, split)) launch(kv_shards ? ca_fwd32_kernel<true, false> : ca_fwd32_kernel<false, false>);
    else if (few) launch(kv_shards ? ca_fwd_kernel<true, true> : ca_fwd_kernel<false, true>);
    else if (geom.merge_tiles > 0) launch(kv_shards ? ca_fwd32_kernel<true, true> : ca_fwd32_kernel<false, true>);
    else launch(kv_shards ? ca_fwd_kernel<true, false> : ca_fwd_kernel<false, false>);
    if (split) hipLaunchKernelGGL(ca_fwd_combine_kernel, cut_grid(split_max_cut(lay.max_blocks, lay.target), p->num_heads_kv, kCutParts), dim3(kCutThreads), 0, s, a);
  }
  return check_launch("ca_fwd");
}
}  // namespace distca
