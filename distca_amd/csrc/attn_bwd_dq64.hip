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

constexpr int kThreads = 256;
constexpr int kRowsWg = 256;            // flattened query rows per workgroup (kDqRows)
constexpr int kKeys = 32;               // keys per tile
constexpr int kRow = 256;               // bytes per tile row, chunks swizzled by tile_swz16
constexpr int kTile = kKeys * kRow;
constexpr int kStageBytes = 2 * kTile;  // K tile, V tile
constexpr int kStages = 4;
constexpr int kLdsRing = kStages * kStageBytes;
constexpr int kRowsLds = 3 * kTile;        // per wave, behind the ring: 32 rows of Q, dO and O on their way in, 64 rows of dQ on their way out
constexpr int kLds = kLdsRing + 4 * kRowsLds;
static_assert(kLds <= 160 * 1024 && kRowsLds >= 64 * kRow, "LDS of a compute unit");
constexpr int kLoadsPerTile = 4;        // vector-memory instructions a wave issues per tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kDoAcc = 2;               // of a wave's four sub-blocks, those whose dO lies in accumulation registers
constexpr int kAhead = 3;               // tiles by which requests run ahead
static_assert(kDqRows == kRowsWg, "the dQ work list is built for blocks of 256 rows");

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// all LDS reads (the compiler knows this form and puts no waits of its own behind it)
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
// The S and dP accumulators are read and overwritten by the vector ALU and must live in vector registers; this file
// is compiled with the compiler's default MFMA form (results in the accumulation registers, right for dQ), so
// these MFMAs are written as assembly.  The compiler does not space such an instruction from the vector
// instructions that read its result (a four-pass MFMA: 8 wait states): the order of a tile's instructions below,
// held in place by the scheduling fences, keeps at least three later MFMAs, each of which waits for the four passes
// of the one before it, between every such MFMA and the first read of its result; a change to the tile body has to keep that.
// The B operands, Q and dO, are in accumulation registers: a wave's 512 registers are 256 of each kind, and the
// vector half is what the tile arithmetic is short of.
typedef float accop_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ accop_t to_acc_regs(elemx8 v) {
  accop_t r;
  asm volatile("; operand to accumulation registers" : "=a"(r) : "0"(__builtin_bit_cast(accop_t, v)));
  return r;
}
__device__ __forceinline__ void mfma16_va(f32x4 &acc, elemx8 a, accop_t b) {  // acc += A B
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %0" : "+v"(acc) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma16_va0(f32x4 &acc, elemx8 a, accop_t b) {  // acc = A B
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma16_a(f32x4 &acc, elemx8 a, elemx8 b) {  // acc += A B, in accumulation registers
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_v(f32x4 &acc, elemx8 a, elemx8 b) {
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_vc(f32x4 &acc, elemx8 a, elemx8 b, const f32x4 &c0) {
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "v"(b), "v"(c0));
}
__device__ __forceinline__ void mfma16_vac(f32x4 &acc, elemx8 a, accop_t b, const f32x4 &c0) {  // acc = A B + c0
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "a"(b), "v"(c0));
}

// SEG: K/V rows are addressed through a table of shards (kv_shards.h) instead of as one dense tensor.
// MERGE: a work item is several consecutive blocks of a task's query rows (sched.h, fwd_merge), worked off one after the
// other; otherwise it is one block.
// SPLIT (batches of few blocks): a work item may be a piece of a block, a range of its K/V tiles (sched.h, piece_count), whose dQ
// goes to a slot; items are taken by workgroup id.
template <bool SEG, bool MERGE, bool SPLIT>
__global__ __launch_bounds__(kThreads, 1) void ca_bwd_dq64_kernel(BwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int nitems = a.sched[0];
  int item, kvh;
  if (!take_item<SPLIT>(a.tickets, nitems, a.hkv, reinterpret_cast<int32_t *>(lds), item, kvh)) return;
  int4 it4 = reinterpret_cast<const int4 *>(a.sched + a.sched_items_off)[item];
  it4.x = uniform_int(it4.x);
  it4.y = uniform_int(it4.y);
  const int task = it4.x;

  // The task's bounds and offsets: every load is issued before the first is used (the optional arrays are read
  // through a pointer that falls back to a place that is always readable, instead of under a branch each: with a
  // branch per array the loads went to memory one after the other, six trips before the kernel could start).
  const int32_t *cq = a.cu_q + task, *ck = a.cu_k + task;
  const int32_t *kvp = a.kv_off ? a.kv_off + task : ck;
  const int64_t *spare = reinterpret_cast<const int64_t *>(a.zero_row);
  const int64_t *qsp = a.qs_task_off ? a.qs_task_off + task : spare, *dqp = a.dq_task_off ? a.dq_task_off + task : spare;
  const int q0_ = cq[0], q1_ = cq[1], k0_ = ck[0], k1_ = ck[1], ks_ = *kvp;
  const int64_t qs_given_ = *qsp, dq_given_ = *dqp;
  fence();
  const int q0 = uniform_int(q0_), q1 = uniform_int(q1_), k0 = uniform_int(k0_), k1 = uniform_int(k1_);
  int ks = uniform_int(ks_);
  const int64_t qs_given = uniform_int64(qs_given_), dq_given = uniform_int64(dq_given_);
  const int64_t qs_task = a.qs_task_off ? qs_given : (int64_t)q0 * a.qs_tok_bytes;
  const int64_t dq_task = a.dq_task_off ? dq_given : (int64_t)q0 * a.dq_tok_bytes;
  const int lq = q1 - q0;
  int lk = k1 - k0;
  const int G = a.group;
  int shift = lk - lq;

  const int nrows = lq * G;
  // the blocks of this item
  int mb_first = it4.y, mb_end = it4.y + 1;
  if constexpr (MERGE) {
    SchedGeom geom;
    geom.rows_per_block = kRowsWg; geom.kv_per_block = kFwdKV; geom.group = G; geom.causal = a.causal; geom.merge_tiles = a.merge_tiles;
    const int m = fwd_merge(geom, lq, lk), nblk = (nrows + kRowsWg - 1) / kRowsWg;
    mb_first = it4.y * m;
    mb_end = mb_first + m < nblk ? mb_first + m : nblk;
  }
  // (a jump back rather than a loop statement: without MERGE the body below is then straight-line code, exactly the
  // kernel that takes one block per item)
  int mblk = mb_first;
  bool requested = false;  // MERGE: the first sub-block's rows of this block are already on their way
next_block:
  // MERGE: the thread index is made opaque once per block, so that what derives from it is computed afresh for every
  // block instead of being carried, and partly spilled, across the whole body
  int tid_ = threadIdx.x;
  if constexpr (MERGE) asm volatile("" : "+v"(tid_));
  const int tid = tid_, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g4 = lane >> 4;
  const int row_wg = mblk * kRowsWg;

  int tok_end = (row_wg + kRowsWg + G - 1) / G;
  if (tok_end > lq) tok_end = lq;
  int nvis = a.causal ? tok_end + shift : lk;
  if (nvis > lk) nvis = lk;
  int ntiles = nvis > 0 ? (nvis + kKeys - 1) / kKeys : 0;
  if constexpr (SPLIT) {
    // A piece is what a whole block over the keys from its first tile on would be: what counts keys from the start of the prefix is
    // moved by the tiles before it.  (The list counts keys in units of kFwdKV.)
    const int w = uniform_int(it4.w);
    int lo, hi;
    piece_range((ntiles * kKeys + kFwdKV - 1) / kFwdKV, item_piece(w), item_pieces(w), a.cut ? uniform_int(a.cut[2]) : 0, &lo, &hi);
    const int end = hi * (kFwdKV / kKeys);
    ntiles = (end < ntiles ? end : ntiles) - lo * (kFwdKV / kKeys);
    ks += lo * kFwdKV;
    lk -= lo * kFwdKV;
    shift -= lo * kFwdKV;
  }

  const uint32_t lds0 = (uint32_t)(uintptr_t)(DISTCA_LDS uint8_t *)lds;
  auto div_group = [&](int n) { return a.group_magic ? (int)__umulhi((uint32_t)n, a.group_magic) : n; };

  // ---- K/V tile fetch: this wave brings rows 8 w .. 8 w + 7 of the K tile and of the V tile, four rows per
  // instruction.  Tiles that lie wholly inside the prefix take a form without per-lane address arithmetic (a scalar
  // base that advances by one tile, per-lane offsets that never change); rows past the prefix read the zero row.
  const int64_t kv_stride = (int64_t)a.hkv * kHeadDim;
  const elem_t *kbase = a.k + (SEG ? 0 : (int64_t)ks * kv_stride) + kvh * kHeadDim;
  const elem_t *vbase = a.v + (SEG ? 0 : (int64_t)ks * kv_stride) + kvh * kHeadDim;
  ShardCursor cur;  // SEG: the shard that holds the rows of the tile requested next
  if constexpr (SEG)
    cur.open(a.shards, SPLIT ? find_shard_wave(a.shards.row_start, a.shards.num_shards, ks) : a.shards.task_shard[task]);
  uint32_t voff[2];
#pragma unroll
  for (int ii = 0; ii < 2; ++ii) {
    const int r = 8 * wave + 4 * ii + (lane >> 4);
    voff[ii] = (uint32_t)((r * kv_stride + (((lane & 15) ^ tile_swz16(r)) * 8)) * 2);
  }
  // SEG: tiles that end at or before key run_lim lie in the present shard, key x of the prefix at kvirt / vvirt +
  // x * kv_stride; a tile past it looks for its shard first, so that a run of tiles inside one shard is requested
  // exactly as tiles of a dense tensor are.
  const elem_t *kvirt = kbase, *vvirt = vbase;
  int run_lim = SEG ? 0 : lk;
  auto issue_whole = [&](uint32_t dst, int j) {
    const elem_t *kt = kvirt + (int64_t)j * kKeys * kv_stride, *vt = vvirt + (int64_t)j * kKeys * kv_stride;
    lds_direct_load16(kt, voff[0], dst);
    lds_direct_load16(kt, voff[1], dst + 4 * kRow);
    lds_direct_load16(vt, voff[0], dst + kTile);
    lds_direct_load16(vt, voff[1], dst + kTile + 4 * kRow);
  };
  auto issue_tile = [&](int stage, int j) {
    const uint32_t dst = lds0 + stage * kStageBytes + 8 * wave * kRow;
    if constexpr (SEG) {
      if ((j + 1) * kKeys <= run_lim) {
        issue_whole(dst, j);
        return;
      }
      const int r0 = ks + j * kKeys;
      cur.seek(a.shards, r0);
      if ((j + 1) * kKeys <= lk && cur.holds(r0, kKeys)) {
        const int64_t back = (int64_t)(cur.lo - ks) * kv_stride * 2;
        kvirt = reinterpret_cast<const elem_t *>(static_cast<uintptr_t>(uniform_i64((int64_t)reinterpret_cast<uintptr_t>(kbase) + cur.k - back)));
        vvirt = reinterpret_cast<const elem_t *>(static_cast<uintptr_t>(uniform_i64((int64_t)reinterpret_cast<uintptr_t>(vbase) + cur.v - back)));
        run_lim = uniform_i32(cur.hi - ks < lk ? cur.hi - ks : lk);
        issue_whole(dst, j);
        return;
      }
#pragma unroll
      for (int ii = 0; ii < 2; ++ii) {
        const int r = 8 * wave + 4 * ii + (lane >> 4);
        const int key = j * kKeys + r;
        const int chunk = (lane & 15) ^ tile_swz16(r);
        const bool ok = key < lk;
        const uint8_t *zero = reinterpret_cast<const uint8_t *>(a.zero_row);
        const uint8_t *kp = ok ? reinterpret_cast<const uint8_t *>(kbase) + shard_row_offset(a.shards, cur, ks + key, 0, kv_stride * 2) : zero;
        const uint8_t *vp = ok ? reinterpret_cast<const uint8_t *>(vbase) + shard_row_offset(a.shards, cur, ks + key, 1, kv_stride * 2) : zero;
        lds_direct_load16_ptr(kp + chunk * 16, dst + 4 * ii * kRow);
        lds_direct_load16_ptr(vp + chunk * 16, dst + kTile + 4 * ii * kRow);
      }
    } else {
      if ((j + 1) * kKeys <= lk) {
        const elem_t *kt = kbase + (int64_t)j * kKeys * kv_stride, *vt = vbase + (int64_t)j * kKeys * kv_stride;
        lds_direct_load16(kt, voff[0], dst);
        lds_direct_load16(kt, voff[1], dst + 4 * kRow);
        lds_direct_load16(vt, voff[0], dst + kTile);
        lds_direct_load16(vt, voff[1], dst + kTile + 4 * kRow);
        return;
      }
#pragma unroll
      for (int ii = 0; ii < 2; ++ii) {
        const int r = 8 * wave + 4 * ii + (lane >> 4);
        const int key = j * kKeys + r;
        const int chunk = (lane & 15) ^ tile_swz16(r);
        const bool ok = key < lk;
        const elem_t *kp = ok ? kbase + (int64_t)key * kv_stride : reinterpret_cast<const elem_t *>(a.zero_row);
        const elem_t *vp = ok ? vbase + (int64_t)key * kv_stride : reinterpret_cast<const elem_t *>(a.zero_row);
        lds_direct_load16_ptr(kp + chunk * 8, dst + 4 * ii * kRow);
        lds_direct_load16_ptr(vp + chunk * 8, dst + kTile + 4 * ii * kRow);
      }
    }
  };

  // The first two tiles are requested before the block's own rows: they land in the ring while the rows pass through
  // the part of LDS behind it.
  if (ntiles > 0) {
    issue_tile(0, 0);
    issue_tile(1, 1);
  }

  // ---- this lane's four rows: Q and dO as B operands (row c16 of a sub-block of 16, d = 32 s + 8 g4 .. +7), statistics
  int row[4], tok[4], lim[4];
  bool valid[4];
  float lse2[4], delta[4];
  accop_t qf[4][4], dof[kDoAcc][4];
  elemx8 dov[4 - kDoAcc][4];
  // The wave's 64 rows of Q, dO and O come through LDS: LDS-direct loads bring four whole rows of 256 bytes per
  // instruction, and the lanes then read their operand fragments (row c16 of a sub-block, chunk 4 s + g4) from there.
  // Loaded straight into the operand layout, every load instruction touched 32 rows, 32 bytes of each, and the address
  // unit takes about a cycle per cache line it has to look up: 48 such loads per wave took 7.7 us to *issue*, a third
  // of what a block of a 1024-token document then spent in its tile loop.  The rows use the 24 KB per wave that lie
  // behind the tile ring (32 rows of Q, dO and O at a time), so the ring is free for the first tiles
  // meanwhile, and each wave reads only what it has loaded itself: no barrier.
  // Before that, and also in one batch, the lse of the lane's four rows (the opaque statements that move Q into the
  // accumulation registers order memory accesses around themselves: no load may be left between them).
  float lse_row[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    row[m] = row_wg + wave * 64 + 16 * m + c16;
    valid[m] = row[m] < nrows;
    // A row past the task (the last block of a task only) reads the task's last row instead, without a branch: with
    // lse2 = +inf its P and dS are zero whatever Q and dO hold, as long as they are finite, and nothing of it is stored.
    const int rc = valid[m] ? row[m] : nrows - 1;
    tok[m] = div_group(rc);
    const int hg = rc - tok[m] * G;
    int lm = a.causal ? tok[m] + shift : lk - 1;
    if (lm > lk - 1) lm = lk - 1;
    lim[m] = lm;
    lse_row[m] = a.lse_tok ? reinterpret_cast<const float *>(a.lse_tok + qs_task + (int64_t)tok[m] * a.qs_tok_bytes)[kvh * G + hg]
                           : a.lse[(int64_t)(kvh * G + hg) * a.total_q + q0 + tok[m]];
  }
  const int wrow0 = row_wg + wave * 64;
  const uint32_t stg = lds0 + kLdsRing + wave * kRowsLds;  // [Q | dO | O] of one half of the wave's rows, 8 KB each
  // requests half m of the wave's rows in block `blk` of the task: instruction i brings rows 32 m + 4 i + lane / 16
  // of the wave, lane % 16 being the position of the 16-byte chunk in the (swizzled) LDS row
  auto request_rows = [&](int blk, int m) {
    const int rw = blk * kRowsWg;
    const int tok0 = div_group(rw);
    const int64_t base = qs_task + (int64_t)tok0 * a.qs_tok_bytes + (int64_t)kvh * G * kHeadDim * 2;
    const uint8_t *qb = reinterpret_cast<const uint8_t *>(a.q) + base, *dob = reinterpret_cast<const uint8_t *>(a.dout) + base,
                  *ob = reinterpret_cast<const uint8_t *>(a.out) + base;
    uint32_t roff[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 32 * m + 4 * i + (lane >> 4);
      int rg = rw + wave * 64 + r;
      if (rg > nrows - 1) rg = nrows - 1;
      const int t = div_group(rg);
      roff[i] = (uint32_t)((t - tok0) * a.qs_tok_bytes + (rg - t * G) * (kHeadDim * 2) + (((lane & 15) ^ tile_swz16(r)) << 4));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) lds_direct_load16(qb, roff[i], stg + i * 4 * kRow);
#pragma unroll
    for (int i = 0; i < 8; ++i) lds_direct_load16(dob, roff[i], stg + kTile + i * 4 * kRow);
#pragma unroll
    for (int i = 0; i < 8; ++i) lds_direct_load16(ob, roff[i], stg + 2 * kTile + i * 4 * kRow);
  };
  const float c = a.scale * kLog2e;
  const int k_rd = c16 * kRow + ((g4 ^ tile_swz16(c16)) << 4);  // A operand rows of a tile, ^ 64*s
  // transposed K operand: lane points at (key 4 g4 + i4 [+ 16], chunk h1 [+ 2 db], half lane & 1)
  const int i4 = (lane & 15) >> 2, h1 = (lane & 3) >> 1;
  const int t_rd = (4 * g4 + i4) * kRow + ((h1 ^ tile_swz16(4 * g4 + i4)) << 4) + 8 * (lane & 1);  // ^ 32*db

  // Absolute LDS addresses of this lane's operand reads in stage 0, the swizzled variants of each read shape,
  // kept in registers: where the stage is a constant (the unrolled loop below) stage and tile sit in the read
  // instruction's offset field and no address arithmetic is left between the MFMAs.
  uint32_t k_ad[4], t_ad[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    t_ad[i] = lds0 + (t_rd ^ (i << 5));
    asm volatile("" : "+v"(t_ad[i]));
    if (i < 4) {
      k_ad[i] = lds0 + (k_rd ^ (i << 6));
      asm volatile("" : "+v"(k_ad[i]));
    }
  }

  f32x4 s0[4], s1[4];        // S, then P, of keys 0 .. 15 and 16 .. 31
  elemx8 fx[4], fy[4];       // K and V fragments of this phase and the next
  auto frag = [&](uint32_t so, int s) { return *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(k_ad[s] + so)); };
  auto x_of = [&](float x, int rb) __attribute__((always_inline)) { return __builtin_fmaf(x, c, -lse2[rb]); };
  auto p_of = [&](float x, int rb) __attribute__((always_inline)) { return fast_exp2(x_of(x, rb)); };
  {
    const uint32_t frag_at = c16 * kRow + ((g4 ^ tile_swz16(c16)) << 4);  // this lane's chunk 0 of row c16; ^ (s << 6)
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      elemx8 qt[2][4], dt[2][4], ot[2][4];
      // MERGE: the first half's rows were requested before the previous block of the item stored its results
      if (m == 0 && !(MERGE && requested)) request_rows(mblk, 0);
      wait_vm<0>();  // (the first tiles, requested before, and lse as well)
      if (m == 0) {  // the first two tiles are there
        fence();
        asm volatile("s_barrier" ::: "memory");
        fence();
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const uint32_t at = stg + 16 * b * kRow + (frag_at ^ (s << 6));
          qt[b][s] = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(at));
          dt[b][s] = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(at + kTile));
          ot[b][s] = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(at + 2 * kTile));
        }
      if (m == 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s) fx[s] = frag(0, s);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are done before the place is filled again
      if (m == 0) request_rows(mblk, 1);   // (they arrive while the first half's sums are made: documents of 128 to 2048 tokens 1 316 us -> 1 307)
      fence();
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int rb = 2 * m + b;
          qf[rb][s] = to_acc_regs(qt[b][s]);
          if (rb < kDoAcc) dof[rb][s] = to_acc_regs(dt[b][s]);
          else dov[rb - kDoAcc][s] = dt[b][s];
        }
      float part[2] = {0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          // (without a tile, of whatever the ring holds, for nothing)
          fence();
          if (s == 0) mfma16_va0(s0[2 * m + b], fx[s], qf[2 * m + b][s]);
          else mfma16_va(s0[2 * m + b], fx[s], qf[2 * m + b][s]);
          fence();
#pragma unroll
          for (int i = 0; i < 8; ++i) part[b] += (float)dt[b][s][i] * (float)ot[b][s][i];
        }
      fence();
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int rb = 2 * m + b;
        delta[rb] = quad_sum(part[b]);  // this lane's quarter of d, then the sum of the four lanes of the row
        lse2[rb] = valid[rb] ? lse_row[rb] * kLog2e : INFINITY;  // rows past the task: P = exp2(-inf) = 0
      }
      if (m == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s0[e >> 2][e & 3] = p_of(s0[e >> 2][e & 3], e >> 2);
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) fy[s] = frag(16 * kRow, s);
  }
  // -delta of the lane's row in all 4 registers of a vector: the C operand of a tile's first dP MFMA, so that
  // dS = P * (what the MFMAs leave) costs one instruction per element
  f32x4 ndl[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) ndl[m] = f32x4{-delta[m], -delta[m], -delta[m], -delta[m]};
  int wrow1 = wrow0 + 63;
  if (wrow1 > nrows - 1) wrow1 = nrows - 1;
  const bool wave_live = wrow0 < nrows;
  int lim_first = 0x7fffffff, lim_last = -1;
  if (wave_live) {
    lim_first = a.causal ? wrow0 / G + shift : lk - 1;
    if (lim_first > lk - 1) lim_first = lk - 1;
    lim_last = a.causal ? wrow1 / G + shift : lk - 1;
    if (lim_last > lk - 1) lim_last = lk - 1;
  }

  f32x4 dqacc[4][8];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int db = 0; db < 8; ++db) dqacc[m][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  // One tile, in six phases of 16 MFMAs.  What a tile begins with is there when it begins: S of its first 16 keys, the exponentials of
  // sub-blocks 0 and 1 of them (kept as they are until the tile is known to be masked), and the K fragments of its other 16 keys.  A MFMA leaves
  // two slots for other instructions, so the arithmetic is spread over all phases: per phase 16, 24, 24, 16, 16, 16 vector instructions, about two behind a MFMA.
  //   1  S, keys 16 .. 31       beside it: P of keys 0 .. 15, sub-blocks 2 and 3; V fragments
  //   2  dP, keys 0 .. 15       P of keys 16 .. 31, sub-blocks 0 to 2; V fragments; then the barrier for the next tile
  //   3  dP, keys 16 .. 31      the rest of P; dS of keys 0 .. 15; the next tile's K fragments
  //   4  S, keys 0 .. 15 of the next tile     dS of keys 16 .. 31, sub-blocks 0 and 1; transposed K fragments
  //   5  dQ, sub-blocks 0 and 1               the rest of dS; transposed K fragments
  //   6  dQ, sub-blocks 2 and 3               P of the next tile, keys 0 .. 15, sub-blocks 0 and 1; its K fragments; request(0 .. 3), the loads
  //                                           of the tile kAhead tiles on, whose stage every wave left before the barrier of phase 2
  // MASKED: the tile straddles the diagonal or the end of the prefix, compare and select per element.
  // Requests are made for tiles below ntiles only (and, in the rounds below, for what lies behind them in the prefix): one past the end, even from
  // the zero row, was waited for in the open before the block's results could leave.  Documents of 256 tokens (65536) 694 us -> 676,
  // of 128 to 2048 1 239 -> 1 220, of 1024 1 033 -> 1 017.
  auto landed = [&](auto two_on) __attribute__((always_inline)) {  // two_on: the tile after the next, or a constant where it is known to be requested
    // the next tile has landed when at most the loads of the one after it are still on their way
    if constexpr (std::is_same_v<decltype(two_on), int>)
      // (the branch is out of the compiler's sight: as one of its own it would end a block of code between the MFMAs)
      asm volatile("s_cmp_lt_i32 %0, %1\n\ts_cbranch_scc1 .Lrequested%=\n\ts_waitcnt vmcnt(0)\n.Lrequested%=:\n\ts_waitcnt vmcnt(%2)" ::"s"(two_on), "s"(uniform_int(ntiles)), "n"(kLoadsPerTile) : "memory", "scc");
    else
      wait_vm<kLoadsPerTile>();
    fence();
    asm volatile("s_barrier" ::: "memory");
    fence();
  };
  // LAST: there is no next tile for this wave, nothing of it is made.
  auto tile = [&](auto stage, auto next_stage, int key0, auto two_on, auto masked, auto last, auto request) __attribute__((always_inline)) {  // stages: ints or constants
    constexpr bool kMasked = decltype(masked)::value, kLast = decltype(last)::value;
    const uint32_t so = (uint32_t)stage * kStageBytes, so_next = (uint32_t)next_stage * kStageBytes;
    f32x4 d0[4], d1[4];  // dP, then dS
    elemx4 ct[8][2];
    auto load_t = [&](int db) {
      ct[db][0] = lds_read_tr(lds_ptr(t_ad[db] + so));
      ct[db][1] = lds_read_tr(lds_ptr(t_ad[db] + so + 16 * kRow));
    };
    // masked: which rows do not see the key of an element, found two elements ahead: a select has to stand two wait states
    // behind its compare (65536 tokens in documents of 128 to 2048, side by side -> ahead: 1 299 us -> 1 280)
    uint64_t hidden[4];
    int last_key[4];  // of this lane's rows, counted from its first key of the tile
    auto find_hidden = [&](int e) __attribute__((always_inline)) {  // element e: keys 16 (e / 16) + e % 4, sub-block e / 4 % 4
      if (e >= 32) return;
      hidden[e & 3] = __builtin_amdgcn_ballot_w64(16 * (e >> 4) + (e & 3) > last_key[(e >> 2) & 3]);
      asm volatile("" : "+s"(hidden[e & 3]));  // here, not where it is used
    };
    // (ahead of the exponential where there is a choice: what follows that one at once has to wait for it)
    auto hide = [&](float x, int e, float hidden_x) __attribute__((always_inline)) {
      if (__builtin_amdgcn_inverse_ballot_w64(hidden[e & 3])) x = hidden_x;
      find_hidden(e + 2);
      return x;
    };
    auto p_elem = [&](int e) __attribute__((always_inline)) {
      const int rb = (e >> 2) & 3, r = e & 3;
      float x = x_of(e < 16 ? s0[rb][r] : s1[rb][r], rb);
      if constexpr (kMasked) x = hide(x, e, -INFINITY);
      x = fast_exp2(x);
      if (e < 16) s0[rb][r] = x;
      else s1[rb][r] = x;
    };
    auto ds_elem = [&](int e) __attribute__((always_inline)) {  // dP accumulated on top of -delta
      const int rb = (e >> 2) & 3, r = e & 3;
      if (e < 16) d0[rb][r] = s0[rb][r] * d0[rb][r];
      else d1[rb][r] = s1[rb][r] * d1[rb][r];
    };
    // dS as B operand: slots 8 g4 .. +3 are keys 4 g4 .. +3, slots 8 g4 + 4 .. +7 the same 16 keys on
    // (pinned where they are made: joined at their MFMA, the two halves would be converted there, with nothing between a conversion and the MFMA)
    u32x2 dsl[4], dsh[4];
    auto pinned = [](f32x4 x) __attribute__((always_inline)) {
      asm volatile("" : "+v"(x));
      u32x2 r = __builtin_bit_cast(u32x2, cvt4(x[0], x[1], x[2], x[3]));
      asm volatile("" : "+v"(r));
      return r;
    };
    auto ds_lo = [&](int rb) __attribute__((always_inline)) { dsl[rb] = pinned(d0[rb]); };
    auto ds_hi = [&](int rb) __attribute__((always_inline)) { dsh[rb] = pinned(d1[rb]); };
    auto ds_frag = [&](int rb) __attribute__((always_inline)) { return cat4(__builtin_bit_cast(elemx4, dsl[rb]), __builtin_bit_cast(elemx4, dsh[rb])); };
    if constexpr (kMasked) {
#pragma unroll
      for (int m = 0; m < 4; ++m) last_key[m] = lim[m] - key0 - 4 * g4;
      find_hidden(0);
      find_hidden(1);
    }
    auto dp_mfma = [&](f32x4 &acc, elemx8 v, int rb, int s) __attribute__((always_inline)) {
      if (rb < kDoAcc) {
        if (s == 0) mfma16_vac(acc, v, dof[rb][s], ndl[rb]);
        else mfma16_va(acc, v, dof[rb][s]);
      } else {
        if (s == 0) mfma16_vc(acc, v, dov[rb - kDoAcc][s], ndl[rb]);
        else mfma16_v(acc, v, dov[rb - kDoAcc][s]);
      }
    };
    // Fragments are requested in the first half of the phase before theirs, so that one wait ahead of a phase does for all of them.
    // ---- phase 1
    wait_lds();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int s = n >> 2, rb = n & 3;
      fence();
      if (s == 0) mfma16_va0(s1[rb], fy[s], qf[rb][s]);
      else mfma16_va(s1[rb], fy[s], qf[rb][s]);
      fence();
      if (kMasked && n < 4) {  // what was made before the tile was known to be masked
        s0[n >> 1][2 * (n & 1)] = hide(s0[n >> 1][2 * (n & 1)], 2 * n, 0.f);
        s0[n >> 1][2 * (n & 1) + 1] = hide(s0[n >> 1][2 * (n & 1) + 1], 2 * n + 1, 0.f);
      }
      if (n < 8 && n % 2 == 0) fx[n / 2] = frag(so + kTile, n / 2);
      if (n > 4 && n < 11 && n % 2 == 1) p_elem(8 + (n - 5) / 2);
      if (n > 10) p_elem(n);
    }
    // ---- phase 2
    wait_lds();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int s = n >> 2, rb = n & 3;
      fence();
      dp_mfma(d0[rb], fx[s], rb, s);
      fence();
      if (n < 8 && n % 2 == 0) fy[n / 2] = frag(so + kTile + 16 * kRow, n / 2);
      if (n < 8 && n % 2 == 1) p_elem(16 + n / 2);
      if (n >= 8) p_elem(12 + n);
    }
    landed(two_on);
    // ---- phase 3
    wait_lds();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int s = n >> 2, rb = n & 3;
      fence();
      dp_mfma(d1[rb], fy[s], rb, s);
      fence();
      if (!kLast && n < 8 && n % 2 == 0) fx[n / 2] = frag(so_next, n / 2);
      // (-delta is kept until here: dead behind a row's last tile, its registers were written over while the MFMA read them as its C operand)
      if (n == 7) asm volatile("" ::"v"(ndl[0]), "v"(ndl[1]), "v"(ndl[2]), "v"(ndl[3]));
      if (n < 8 && n % 2 == 1) p_elem(28 + n / 2);
      if (n >= 8) ds_elem(2 * n - 16), ds_elem(2 * n - 15);
    }
    // ---- phase 4
    wait_lds();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int s = n >> 2, rb = n & 3;
      fence();
      if constexpr (!kLast) {
        if (s == 0) mfma16_va0(s0[rb], fx[s], qf[rb][s]);
        else mfma16_va(s0[rb], fx[s], qf[rb][s]);
      } else if (n < 4) {
        asm volatile("s_nop 3");  // (in the place of four MFMAs between dP's and the first read of it)
      }
      fence();
      if (n < 11 && n % 2 == 0) load_t(n / 2);
      if (n == 1 || n == 3) ds_elem(15 + n), ds_elem(16 + n);
      if (n == 5) ds_lo(0);
      if (n == 7) ds_hi(0);
      if (n == 9 || n == 11) ds_elem(11 + n), ds_elem(12 + n);
      if (n == 12) ds_lo(1);
      if (n == 13) ds_hi(1);
      if (n == 14) ds_lo(2);
      if (n == 15) ds_lo(3);
    }
    // ---- phase 5.  Consecutive MFMAs share an operand, here and in phase 6: what an operand costs in power is its change.
    wait_lds();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int db = n >> 1, rb = (n ^ db) & 1;
      if (n == 12) wait_lds();
      const elemx8 kt = cat4(ct[db][0], ct[db][1]);
      fence();
      mfma16_a(dqacc[rb][db], kt, ds_frag(rb));
      fence();
      if (n < 2) load_t(6 + n);
      if (n == 2 || n == 4) ds_elem(22 + n), ds_elem(23 + n);
      if (n == 6) ds_hi(2);
      if (n == 8 || n == 10) ds_elem(20 + n), ds_elem(21 + n);
      if (n == 12) ds_hi(3);
    }
    // ---- phase 6
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int db = 7 - (n >> 1), rb = 2 + ((n ^ (n >> 1)) & 1);
      const elemx8 kt = cat4(ct[db][0], ct[db][1]);
      fence();
      mfma16_a(dqacc[rb][db], kt, ds_frag(rb));
      fence();
      if (n % 4 == 0) request(n / 4);
      if constexpr (!kLast) {
        if (n < 8 && n % 2 == 1) fy[n / 2] = frag(so_next + 16 * kRow, n / 2);
        const int e = n == 2 ? 0 : n == 6 ? 1 : n == 9 ? 2 : n == 10 ? 3 : n == 11 ? 4 : n >= 13 ? n - 8 : -1;
        if (e >= 0) s0[e >> 2][e & 3] = p_of(s0[e >> 2][e & 3], e >> 2);
      }
    }
  };

  // Tiles are walked from key 0 up, so the first key of a tile only grows: first come tiles that every row of the
  // wave sees whole (no masking), then tiles on the diagonal or at the end of the prefix (masked), then, for waves
  // whose rows end below those of the block's last wave, tiles that none of their rows sees.  Each kind has a loop
  // of its own with one body; every wave passes the same barriers and makes the same requests in all of them.
  int p = 0;
  static_assert(kAhead == 3, "two tiles came in with the rows; stage (p + 3) % 4 is the one that tile p - 1 has left");
  if (ntiles > 2) issue_tile(2, 2);
  auto none = [](int) {};
  auto issue_ahead = [&](int j) __attribute__((always_inline)) {
    if (j < ntiles) issue_tile(j % kStages, j);
  };
  const uint32_t dst_w = lds0 + 8 * wave * kRow;
  // four unmasked tiles per round, one per ring stage, as long as the fourth is still unmasked and the tiles requested meanwhile lie
  // wholly inside the prefix (SEG: and in the present shard; the loop of single tiles comes back to this one behind every shard's end: tick of
  // 16384 tokens 1 864 us -> 1 817, tick over a document of 131072 tokens 36 870 -> 35 940, with requests behind the barrier before)
  int whole_end = wave_live ? (lim_first + 1) / kKeys : 0;  // the tiles that every row of the wave sees whole
  whole_end = uniform_int(whole_end < ntiles ? whole_end : ntiles);
  auto rounds = [&]() __attribute__((always_inline)) {
    for (; p + 4 <= whole_end && (p + 4 + kAhead) * kKeys <= (SEG ? run_lim : lk); p += 4) {
      auto four = [&](auto st) __attribute__((always_inline)) {
        constexpr int kSt = decltype(st)::value;
        using Next = std::integral_constant<int, (kSt + 1) % kStages>;
        const int64_t at = (int64_t)(p + kSt + kAhead) * kKeys * kv_stride;
        const elem_t *kt = (SEG ? kvirt : kbase) + at, *vt = (SEG ? vvirt : vbase) + at;
        const uint32_t dst = dst_w + ((kSt + kAhead) % kStages) * kStageBytes;
        tile(st, Next{}, (p + kSt) * kKeys, std::true_type{}, std::false_type{}, std::false_type{}, [&](int i) __attribute__((always_inline)) {
          lds_direct_load16(i < 2 ? kt : vt, voff[i & 1], dst + (i >> 1) * kTile + (i & 1) * 4 * kRow);
        });
      };
      four(std::integral_constant<int, 0>{});
      four(std::integral_constant<int, 1>{});
      four(std::integral_constant<int, 2>{});
      four(std::integral_constant<int, 3>{});
    }
  };
  if constexpr (!SEG) rounds();
  for (; p < whole_end; ++p) {
    if constexpr (SEG) {
      if (p % kStages == 0) {
        rounds();
        if (p >= whole_end) break;
      }
    }
    tile(p % kStages, (p + 1) % kStages, p * kKeys, p + 2, std::false_type{}, std::false_type{}, none);
    issue_ahead(p + kAhead);
  }
  int seen_end = lim_last / kKeys + 1;  // the tiles that some row of the wave sees
  seen_end = uniform_int(!wave_live || lim_last < 0 ? 0 : seen_end < ntiles ? seen_end : ntiles);
  for (; p < seen_end - 1; ++p) {
    tile(p % kStages, (p + 1) % kStages, p * kKeys, p + 2, std::true_type{}, std::false_type{}, none);
    issue_ahead(p + kAhead);
  }
  if (p < seen_end) {
    tile(p % kStages, (p + 1) % kStages, p * kKeys, p + 2, std::true_type{}, std::true_type{}, none);
    issue_ahead(p + kAhead);
    ++p;
  }
  for (; p < ntiles; ++p) {
    landed(p + 2);
    issue_ahead(p + kAhead);
  }
  wait_vm<0>();  // nothing may still be on its way into LDS when the workgroup ends

  // MERGE: the next block's first rows are requested now and arrive while this block's results are stored; the dQ rows
  // then leave through the wave's stage of the ring, which every wave has left (the barrier), instead of through the
  // rows' place.
  if constexpr (MERGE) {
    requested = mblk + 1 < mb_end;
    __syncthreads();
    if (requested) request_rows(mblk + 1, 0);
  }

  // ---- epilogue: the row statistics for the dK/dV kernel, which runs after this one (stored here rather than where
  // they are made: the wait that precedes the tile loop would have to see the stores through as well), and the dQ rows.
  // A lane holds a quarter of each of its four rows in pieces of 8 bytes (block db holds d = 16 db + 4 g4 .. +3):
  // stored from there, an instruction touched 16 rows.  The pieces go to the wave's 16 KB behind the ring instead, in
  // the tiles' swizzled row layout, and leave from there four whole rows per instruction.
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    if (valid[m] && g4 == 0) {
      const int hg = row[m] - tok[m] * G;
      const int64_t so = (int64_t)(kvh * G + hg) * a.total_q + q0 + tok[m];
      a.lse2_w[so] = lse2[m];
      a.dscaled_w[so] = ndl[m][0];  // -delta: the start value of the dP accumulators in the dK/dV kernel
    }
  }
  if constexpr (SPLIT) {
    // a piece's dQ where the kernel that adds up reads it (cut_blocks.h): d0 = 16 db + 4 g4 of row r of the wave at part r / 32,
    // d block db % 4, quarter 2 (db / 4) + g4 / 2, lane 32 (g4 % 2) + r % 32
    const int slot = a.slot ? uniform_int(a.slot[2 * item]) : -1;
    if (slot >= 0) {
      f32x4 *op = reinterpret_cast<f32x4 *>(a.partial + ((int64_t)slot * a.hkv + kvh) * kDqSlotBytes) + wave * 32 * 64 + (g4 >> 1) * 64 + (g4 & 1) * 32 + c16;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int db = 0; db < 8; ++db) op[(16 * (m >> 1) + 4 * (db & 3) + 2 * (db >> 2)) * 64 + 16 * (m & 1)] = dqacc[m][db];
      return;
    }
  }
  {
    const uint32_t out_b = MERGE ? lds0 + wave * kStageBytes : stg;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int db = 0; db < 8; ++db)
        *static_cast<DISTCA_LDS elemx4 *>(const_cast<DISTCA_LDS void *>(
            lds_ptr(out_b + (16 * m + c16) * kRow + (((2 * db + (g4 >> 1)) ^ tile_swz16(c16)) << 4) + 8 * (g4 & 1)))) =
            cvt4(dqacc[m][db][0] * a.scale, dqacc[m][db][1] * a.scale, dqacc[m][db][2] * a.scale, dqacc[m][db][3] * a.scale);
    // (LDS operations of one wave complete in order: the reads below see the writes above)
    uint8_t *dq_blk = reinterpret_cast<uint8_t *>(a.dq) + dq_task + (int64_t)kvh * G * kHeadDim * 2;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 4 * i + (lane >> 4);
      const int rg = wrow0 + r;
      const elemx8 v = *static_cast<const DISTCA_LDS elemx8 *>(lds_ptr(out_b + r * kRow + ((lane & 15) << 4)));
      if (rg < nrows) {
        const int t = div_group(rg);
        *reinterpret_cast<elemx8 *>(dq_blk + (int64_t)t * a.dq_tok_bytes + (rg - t * G) * (kHeadDim * 2) + (((lane & 15) ^ tile_swz16(r)) << 4)) = v;
      }
    }
  }
  if constexpr (MERGE) {
    if (++mblk < mb_end) {
      __syncthreads();  // every wave has left the ring's stages before the next block's first tiles are requested
      goto next_block;
    }
  }
}

// Adds up the pieces of the blocks that were cut, in their order (cut_blocks.h).
__global__ __launch_bounds__(kCutThreads) void ca_bwd_dq64_combine_kernel(BwdArgs a) {
  const int kvh = blockIdx.y, sub = blockIdx.z, lane = threadIdx.x & 63, db = threadIdx.x >> 6, G = a.group;   // sub: two of a wave, four waves
  add_up_cut_blocks(
      a.cut,
      [&](const int4 &e, f32x4 (&o)[4]) {
        const f32x4 *first = reinterpret_cast<const f32x4 *>(a.partial + ((int64_t)e.w * a.hkv + kvh) * kDqSlotBytes);
        add_pieces(first + (16 * sub + 4 * db) * 64 + lane, a.hkv * (kDqSlotBytes / 16), 64, e.z, o);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[k][r] *= a.scale;
      },
      [&](const int4 &e, int r) -> elem_t * {
        const int q0 = a.cu_q[e.x], nrows = (a.cu_q[e.x + 1] - q0) * G, row = e.y * kRowsWg + 32 * sub + r;
        if (row >= nrows) return nullptr;
        const int tok = row / G, hg = row - tok * G;
        return reinterpret_cast<elem_t *>(reinterpret_cast<uint8_t *>(a.dq) + (a.dq_task_off ? a.dq_task_off[e.x] : (int64_t)q0 * a.dq_tok_bytes) +
                                          (int64_t)tok * a.dq_tok_bytes) + (kvh * G + hg) * kHeadDim;
      });
}

}  // namespace

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
  if (max_cut > 0) hipLaunchKernelGGL(ca_bwd_dq64_combine_kernel, cut_grid(max_cut, a.hkv, kCutParts), dim3(kCutThreads), 0, stream, a);
  return DISTCA_OK;
}

}  // namespace distca
