// Tile geometry of the attention kernels and the checks every entry point shares.
#pragma once
#include <math.h>
#include <stdlib.h>

#include "api_util.h"
#include "kv_shards.h"
#include "sched.h"

namespace distca {

constexpr int kHeadDim = 128;

// Forward kernel: each wave owns 32 flattened query rows, two sub-blocks of 16; KV tiles of 64 keys.  That
// keeps a wave under 256 registers, so a compute unit holds eight waves.
constexpr int kFwdWaves = 8;  // waves per workgroup of the forward kernel
constexpr int kFwdRows = kFwdWaves * 32;
constexpr int kDqRows = 256;  // the dQ kernel: four waves of four 16-row sub-blocks
constexpr int kFwdKV = 64;

// dK/dV kernel: a workgroup owns 256 keys (four waves of 64, one per SIMD); query rows are streamed in blocks of
// 32 flattened rows.
constexpr int kBwdRows = 32;
constexpr int kBwdKV = 256;
// A piece's slot: the accumulators of a dQ block (256 rows) or of a key block (dK and dV of 256 keys) as they lie
constexpr int64_t kDqSlotBytes = (int64_t)kDqRows * kHeadDim * 4, kDkdvSlotBytes = 2 * (int64_t)kBwdKV * kHeadDim * 4;

inline int validate_params(const distca_ca_params *p) {
  if (p->head_dim != kHeadDim) return fail(DISTCA_E_UNSUPPORTED, "head_dim=%d: the kernels are built for head_dim 128 (smaller ones can be zero-padded to it)", p->head_dim);
  if (p->dtype != 0 && p->dtype != DISTCA_DTYPE_BF16 && p->dtype != DISTCA_DTYPE_F16)
    return fail(DISTCA_E_UNSUPPORTED, "dtype=%d: the attention kernels take bf16 (%d, or 0) or fp16 (%d) elements", p->dtype, DISTCA_DTYPE_BF16, DISTCA_DTYPE_F16);
  if (p->num_heads_q <= 0 || p->num_heads_kv <= 0 || p->num_heads_q % p->num_heads_kv)
    return fail(DISTCA_E_INVALID, "num_heads_q=%d must be a positive multiple of num_heads_kv=%d", p->num_heads_q, p->num_heads_kv);
  if (p->num_heads_kv > kSchedMaxHeads) return fail(DISTCA_E_UNSUPPORTED, "num_heads_kv=%d: at most %d kv heads", p->num_heads_kv, kSchedMaxHeads);
  if (p->num_tasks < 0 || p->total_q < 0 || p->total_k < 0 || p->max_seqlen_q < 0 || p->max_seqlen_k < 0)
    return fail(DISTCA_E_INVALID, "negative size in distca_ca_params");
  if (!(p->softmax_scale > 0.f) || !isfinite(p->softmax_scale)) return fail(DISTCA_E_INVALID, "softmax_scale must be positive and finite");
  const int64_t group = p->num_heads_q / p->num_heads_kv;
  if ((int64_t)p->max_seqlen_q * group >= (1ll << 30) || (int64_t)p->total_q * group >= (1ll << 31))
    return fail(DISTCA_E_INVALID, "query rows x heads-per-group exceeds 32-bit tile indexing");
  return DISTCA_OK;
}

// Batches of short tasks have the forward and dQ kernels work off several consecutive blocks of a task per work item
// (sched.h, fwd_merge).  Whether a batch is one is decided from host-known sizes, the mean task length: the kernels
// built for merged items carry a loop around their body, which the ones for long tasks are spared.
#ifndef DISTCA_MERGE_MEAN_TOKENS
#define DISTCA_MERGE_MEAN_TOKENS 2048
#endif
constexpr int32_t kMergeMeanTokens = DISTCA_MERGE_MEAN_TOKENS;  // batches whose tasks average fewer query tokens than this
#ifndef DISTCA_MERGE_TILES_FWD
#define DISTCA_MERGE_TILES_FWD 128
#endif
constexpr int32_t kMergeTilesFwd = DISTCA_MERGE_TILES_FWD;  // KV tiles (of 64 keys) a merged forward item aims for
#ifndef DISTCA_MERGE_TILES_DQ
#define DISTCA_MERGE_TILES_DQ 128
#endif
constexpr int32_t kMergeTilesDq = DISTCA_MERGE_TILES_DQ;    // the same for a merged dQ item (its list counts keys in the same unit)
inline bool merge_short_tasks(const distca_ca_params *p) {
  return p->num_tasks > 0 && (int64_t)p->total_q < (int64_t)kMergeMeanTokens * p->num_tasks;
}
// The lists as they are launched: merging trades workgroups for the fixed part of a block, which pays only where the blocks
// fill the device many times over, the more so the longer the tasks: from 8 blocks of query rows per compute unit on where they average
// fewer than kMergeShortMeanTokens, else from 12 on.  The former's items aim for 64 tiles, and for 32 below 16 blocks per unit.  us,
// forward and backward of documents of 64 to n tokens, 32/8 heads, with no merging / 32 / 64 / 128 tiles an item: n = 1024, 9 blocks per
// unit 766 / 726 / 746 / 805, 16 blocks 1325 / 1266 / 1260 / 1352, 32 blocks 2624 / 2514 / 2446 / 2578, 64 blocks 5364 / 4974 / 4835 /
// 4920; n = 512, 32 blocks 2194 / 2045 / 1992 / 2016.  At n = 2048 (1056 tokens in the mean) 64 tiles lose to 128 by 1 % from 24
// blocks per unit on, and at n = 3500 all are within 1 %.  Below 8 blocks the kernels are those for few items (few_row_blocks), which
// do not merge.  num_heads_q / num_heads_kv cancel: blocks x kv heads = total_q * Hq / rows.
constexpr int32_t kMergeShortMeanTokens = 768;
inline SchedGeom launched_geom(SchedGeom g, const distca_ca_params *p) {
  const int64_t blocks = (int64_t)p->total_q * p->num_heads_q, per_cu = (int64_t)g.rows_per_block * num_compute_units();
  const bool very_short = (int64_t)p->total_q < (int64_t)kMergeShortMeanTokens * p->num_tasks;
  if (blocks < (very_short ? 8 : 12) * per_cu) g.merge_tiles = 0;
  else if (very_short) g.merge_tiles = blocks < 16 * per_cu ? 32 : 64;   // (these average below kMergeMeanTokens: merge_tiles was set)
  return g;
}
inline SchedGeom fwd_geom(const distca_ca_params *p) {
  SchedGeom g;
  g.split_target = 0;
  g.min_piece = kMinPiece;
  g.units_per_head = g.item_cost = g.piece_extra = g.add_cost = 0;
  g.beside = 0.f;
  g.walk_round = 0;
  g.merge_tiles = merge_short_tasks(p) ? kMergeTilesFwd : 0;
  g.rows_per_block = kFwdRows;
  g.kv_per_block = kFwdKV;
  g.group = p->num_heads_q / p->num_heads_kv;
  g.causal = p->causal != 0;
  const int64_t worst = (int64_t)p->max_seqlen_k / kFwdKV + 1;
  g.cost_shift = pick_cost_shift(worst > g.merge_tiles ? worst : g.merge_tiles);
  return g;
}
// Key blocks are cut into pieces (sched.h) when the batch has so few of them that they could not occupy the
// device twice over.  Returns the number of pieces to aim for per kv head, 0 = no cutting.  A caller that asks for a
// deterministic backward and brings the smallest workspace gets whole blocks (the same bits either way: pieces are added up in
// their order), one that does not brings room for a few pieces (bwd_small_pieces_bytes).
constexpr int kSplitPiecesPerCU = 2;
// Upper bounds, from host-known sizes, of the number of key blocks = sum over tasks of ceil(Lk / kBwdKV).
// When every task has its own K/V rows the Lk add up to total_k at most; when tasks read shared rows
// (kv_task_offsets) only Lk <= max_seqlen_k is known.
inline int64_t bwd_key_blocks_own_rows(const distca_ca_params *p) { return (int64_t)p->total_k / kBwdKV + p->num_tasks + 1; }
inline int64_t bwd_key_blocks_bound(const distca_ca_params *p) {
  const int64_t by_total = bwd_key_blocks_own_rows(p);
  const int64_t by_max = ((int64_t)p->max_seqlen_k / kBwdKV + 1) * p->num_tasks + 1;
  return by_total > by_max ? by_total : by_max;
}
inline bool few_key_blocks(const distca_ca_params *p, int per_cu) {
  // (compute units of the current device; 256 when there is none, the host mirror on a CPU box)
  return bwd_key_blocks_own_rows(p) * p->num_heads_kv < (int64_t)per_cu * num_compute_units();
}
constexpr int kSplitFewPerCU = 2, kSplitPreferredPerCU = 8;
// (`per_cu`: below how many blocks per compute unit)
inline int32_t bwd_split_pieces(const distca_ca_params *p, int per_cu, int min_piece) {
  const int cus = num_compute_units();
  if (!few_key_blocks(p, per_cu)) return 0;
  const int64_t t = kSplitPiecesPerCU * cus / p->num_heads_kv;
  // (no more than there can be: every block in pieces of min_piece)
  const int64_t rows = (int64_t)p->total_q * (p->num_heads_q / p->num_heads_kv);
  const int64_t all = bwd_key_blocks_bound(p) * ((rows / kBwdRows + p->num_tasks + min_piece) / min_piece);
  return (int32_t)(t < 1 ? 1 : (t < all ? t : all));
}
inline int32_t preferred_key_pieces(const distca_ca_params *p) { return bwd_split_pieces(p, kSplitPreferredPerCU, kMinPieceWorth); }
// What the smallest workspace of a small batch with deterministic == 0 holds beside the lists and the row statistics: 8 bytes per
// stored element of K, which callers with a buffer of their own have always brought (they once were fp32 accumulators of dK and dV).
inline bool bwd_small_pieces(const distca_ca_params *p) { return !p->deterministic && few_key_blocks(p, kSplitFewPerCU); }
inline int32_t bwd_small_list_pieces(const distca_ca_params *p) {   // ... and the room its dK/dV list has beside the blocks
  const int32_t t = kSplitPiecesPerCU * num_compute_units() / p->num_heads_kv;
  return t > 0 ? t : 1;
}
inline int64_t bwd_small_pieces_bytes(const distca_ca_params *p) {
  return 2 * (((int64_t)p->total_k * p->num_heads_kv * kHeadDim * 4 + 255) / 256 * 256);
}
// The pieces aimed for there: as many as leave the slots and tables of the worst case room (the longest blocks of a batch of unequal
// documents; one document alone has no block of twice the average cost, and stays whole).
inline int32_t bwd_split_target(const distca_ca_params *p) {
  if (!bwd_small_pieces(p)) return 0;
  const int64_t blocks = bwd_key_blocks_bound(p);
  const int32_t list = bwd_small_list_pieces(p), t = bwd_split_pieces(p, kSplitFewPerCU, kMinPiece);
  const int64_t slots = (bwd_small_pieces_bytes(p) - split_tables_bytes(blocks, list, blocks + list)) / (kDkdvSlotBytes * p->num_heads_kv);
  return slots < 2 ? 0 : (int32_t)(slots / 2 < t ? slots / 2 : t);
}
// Blocks of query rows are cut into pieces of consecutive KV tiles when the batch has so few of them that the longest one
// could bound the launch: fewer than kSplitMaxBlocksPerCU blocks per compute unit (above that longest-first dispatch evens
// them out), and more than kCutFromTiles* KV tiles that cutting could take off the longest block (row_tiles_to_gain).
// Below the line the second launch, which takes 4.5 us though nothing be cut, and the pieces' own time cost more than they give: us
// forward, cut / whole: 1100 tokens at 4/1 heads (17 tiles to gain) 29.2 / 24.5, 4 x 1024 at 8/2 (15) 33.7 / 24.8, 1500 at 32/8 (15) 40.9 / 32.5,
// 2048 at 32/8 (16) 55 / 52, 2560 + 1024 + 512 at 32/8 (15) 75.5 / 71.2, 4096 at 32/8 (0) 129 / 125, 12000 at 32/8 (0) 934 / 926; above it: 2048 at 8/2 (29)
// 38.1 / 39.5, 2048 at 4/1 (31) 34.2 / 39.0, 3000 at 4/1 (42) 41.5 / 54.2, 8192 at 8/2 (64) 145 / 159.
// dQ's tiles are longer, its line lower: us backward, dQ cut / whole: 1100 at 32/8 (13.2) 102.7 / 100.0, 4 x 1024 at 8/2 (15) 102.5 / 98.7, 1500 at 32/8 (15.2)
// 127.7 / 124.8, 2560 + 1024 + 512 at 32/8 (15) 233.8 / 231.3; at it, by heads: 1024 at 8/2 (15.9) 76.5 / 81.5, 2048 at 32/8 (16.5) 167.7 / 164.6; above it: 1100 at
// 8/2 (16.8) 79.1 / 87.1, 1100 at 4/1 (17.4) 75.0 / 86.1, 2048 at 8/2 (29) 97.1 / 123.5.
// Returns the number of pieces to aim for per kv head, 0 = no cutting.
// It depends only on sizes that do not change with how K/V are stored, so that a tick gives the same bits in every form.
constexpr int kSplitRowPiecesPerCU = 2;
constexpr int kSplitMaxBlocksPerCU = 8;
constexpr int kCutFromTilesFwd = 24, kCutFromTilesDq = 16;
inline bool few_row_blocks(const distca_ca_params *p) {
  return (int64_t)p->total_q * p->num_heads_q < (int64_t)kSplitMaxBlocksPerCU * kFwdRows * num_compute_units();
}
// Whether a forward of few blocks has 32x32x16 MFMAs (attn_fwd32.inc) rather than 16x16x32 (attn_fwd.hip).  The smaller ones save energy and cost cycles, so
// they are for what runs long enough at full load to be bound by power.  That is not so up to prefixes of kFwd32Keys, whose blocks are short, up to
// kFwd32Tiles tiles a compute unit, as far as the bounds tell, nor, up to kFwd32TilesOnce of them and prefixes of kFwd32KeysOnce, where every unit has a block at
// most: half of them are soon done.  us forward, 16x16x32 / 32x32x16 (tiles a unit): 200 tokens at 4/1 heads 11.3 / 10.3, 600 18.8 / 16.5, 1500 (9) at 4/1 34.4 / 30.1, at 32/8
// 36.2 / 32.2, 2048 (17) at 32/8 48.8 / 45.9, 2500 (24) 61.2 / 59.9, 256 rows to 8192 at 8/2 40.1 / 37.6, 4096 in pieces (17) at 8/2 60.9 / 59.9, 5000 (24) 73.3 / 73.1,
// 12 x 1024 (51) at 32/8 127.2 / 125.1, a block a unit, 4096 (33) at 16/4 97.5 / 91.9, 8 x 2048 (17) at 4/1 57.9 / 54.8; on the other side 1800 (25) at 64/8 57.6 / 57.8,
// 6000 in pieces (34) at 8/2 91.6 / 92.3, 8192 (32) at 4/1 89.1 / 90.0, 3 x 5000 (37) 91.7 / 92.9, 3000 (35) at 32/8 74.2 / 76.2, 2 x 2048 (33) 67.7 / 69.3, 10 x 1500 (91)
// 208.5 / 208.5, 4096 (66) 119.3 / 124.0, 8192 434 / 454.
// Where blocks stay whole for want of room for pieces (split: there is) and no unit has two, most units are idle however long they are: 8192 at 4/1 154 / 135, 6000 at 8/2
// 116 / 105, 8 x 512 rows to 32768 at 4/1 590 / 510, 8192 (a block for every unit) at 8/2 162 / 159.
// As row_split_target it must not know how K/V are stored.
constexpr int kFwd32Keys = 1280, kFwd32Tiles = 24, kFwd32KeysOnce = 4096, kFwd32TilesOnce = 33;
inline bool fwd_mfma32(const distca_ca_params *p, bool split) {
  const int64_t k = p->max_seqlen_k, q = p->max_seqlen_q < k ? p->max_seqlen_q : k, rows = (int64_t)p->total_q * p->num_heads_q, units = num_compute_units();
  const bool one_each = rows <= kFwdRows * units, once = one_each && k <= kFwd32KeysOnce;
  if (k <= kFwd32Keys || (one_each && !split)) return true;
  const int64_t keys = p->causal ? k - q / 2 : k;   // that a row sees on average, of a task with the longest prefix
  return rows * keys <= (int64_t)(once ? kFwd32TilesOnce : kFwd32Tiles) * kFwdRows * kFwdKV * units;
}
// dQ and dK/dV side by side in one launch (attn_bwd_pair.hip) up to kPairBlocksPerCU blocks of query rows per compute unit: each then
// fills what the other's longest blocks leave idle, and a launch is saved.  Beyond that their last blocks are a small part of the time and the pass over dO
// and O that makes the row statistics ahead of both shows.  us backward, one after the other / side by side: 256 tokens at 8/2 heads 51 / 34, 389 at 4/1
// 56 / 36, 1000 at 4/1 79 / 55, 2048 at 4/1 (both cut) 88 / 64, 8 x 1000 at 32/8 299 / 261, 8192 at 8/2 458 / 395, 4 x 2300 at 32/8 593 / 507, 2 x 4096 at 32/8 775 / 718; at 4 blocks a
// unit 8192 at 32/8 1404 / 1354, 32768 at 8/2 5276 / 5123; at 5 10000 at 32/8 2040 / 2010, 40000 at
// 8/2 7929 / 7718; at 6 12000 at 32/8 2772 / 2821, at 8 4 x 4000 at 32/8 1329 / 1364.
constexpr int kPairBlocksPerCU = 5;
// What either list's items take of the other's time: 256 rows by 64 keys of dQ 2.1 us, the same area as two blocks of dK/dV at 1.35, hence 0.78 of
// dQ's beside dK/dV and 1.28 the other way round; somewhat less packs better (sched.h, pieces_time; dQ's blocks of one document that has few of them in
// smaller pieces).
constexpr float kDqBesideDkdv = 0.7f, kDkdvBesideDq = 0.68f;
constexpr int32_t kMinPieceBeside = 11;   // of dK/dV (8 in its place: 1024 tokens at 8/2 heads 56 us for 54, 14: 1100 56 for 54)
// Whether the slots of both kernels' pieces lie side by side, as they have to where both are written at a time: within what a preferred workspace has at
// most for slots.
inline bool slots_apart(const distca_ca_params *p, int64_t blocks_kv, int32_t target_kv, int64_t blocks_q, int32_t target_q) {
  return (split_max_slots(blocks_kv, target_kv) * kDkdvSlotBytes + split_max_slots(blocks_q, target_q) * kDqSlotBytes) * p->num_heads_kv <= 1024 * kDkdvSlotBytes;
}
// An upper bound, times *scale, of the KV tiles that cutting could take off the longest block of query rows: all of its tiles but the load of a
// unit, of which only the part counts that the task of the longest prefix brings along, half of its tiles for every block of that task per unit
// (from two blocks per unit on pieces, of which there are two a unit, are on average no shorter than the task's blocks: asked, the list builder cuts none of such a task).  How many rows that task has is known where it is the only one, and
// where the tasks are whole documents, which equal bounds within the batch's tokens are taken for: of all lengths up to the bound, which need
// not be reached, a document of one block per unit has the most to gain.  Otherwise the most rows may be one task's and the longest
// prefix another's, a new document's and a short shard's at the end of a long one; then all tiles count, and the list builder, which sees
// the tasks, decides.  us at 32/8 heads with the one task's rows set against the other's prefix / left to the builder, forward, backward:
// 4096 + 256 rows over 4096 + 131072 keys 2175 / 646, 4915 / 2235; 5000 + 300 + 2000 over 5000 + 60000 + 8000 1104 / 653, 2998 / 2183.
// And at 8/2 heads, the bound taken for a length / for a bound: 8192 + 16 x 512 tokens, bounds of 16384, 173 / 169, 570 / 534.  What the second launch
// costs where the bound is reached and longest-first would have done: 16384 + 2000 tokens 481 / 484, 1672 / 1675.
inline int64_t row_tiles_to_gain(const distca_ca_params *p, int64_t *scale) {
  const int64_t heads = p->num_heads_q, two_each = 2 * (int64_t)kFwdRows * num_compute_units();   // rows x heads of two blocks per unit
  const bool alone = p->num_tasks == 1, documents = p->max_seqlen_q == p->max_seqlen_k && p->max_seqlen_k <= p->total_q;
  int64_t tiles = (int64_t)p->max_seqlen_k / kFwdKV + 1, tokens = 0;
  if (alone || documents) {
    tokens = p->max_seqlen_q < p->max_seqlen_k ? p->max_seqlen_q : p->max_seqlen_k;   // (queries beyond the keys see nothing)
    if (tokens > p->total_q) tokens = p->total_q;
    if (!alone && 2 * tokens * heads > two_each) tokens = two_each / 2 / heads, tiles = tokens / kFwdKV;
  }
  *scale = two_each;
  return tokens * heads < two_each ? tiles * (two_each - tokens * heads) : 0;
}
inline int32_t row_split_target(const distca_ca_params *p, int64_t max_blocks, int from_tiles) {
  if (!few_row_blocks(p)) return 0;
  int64_t scale;
  if (row_tiles_to_gain(p, &scale) <= from_tiles * scale) return 0;
  const int64_t tiles = (int64_t)p->max_seqlen_k / kFwdKV + 1;
  const int64_t most = (tiles + kMinPieceWorth - 1) / kMinPieceWorth;   // pieces of the longest block
  const int64_t t = kSplitRowPiecesPerCU * num_compute_units() / p->num_heads_kv, all = max_blocks * most;
  return (int32_t)(t < 1 ? 1 : (t < all ? t : all));
}
// Workgroups for a list: 5/4 of its places, drawing tickets (sched.h, take_item), or, where the items are few, one each.
inline int64_t list_grid(const distca_ca_params *p, int64_t items, bool few) {
  return few ? items * p->num_heads_kv : items * p->num_heads_kv * kSchedOversubNum / kSchedOversubDen;
}
// A list of which only what is worth it is cut (sched.h, worth_cutting).  item_cost and piece_extra in the list's cost unit: an
// item's ticket, first loads and last stores take 11 us against 1.7 us per forward tile (dQ 15 against 2.4, dK/dV 14 against 1.5
// per query block, with 32x32x16 MFMAs; with 16x16x32 ones, one item a unit, a tile of dQ takes 2.1 us and a block of dK/dV 1.35, 2.3 and 1.55 before: the
// costs below were left, which makes an item look a tenth cheaper than it is), a piece's fp32 result written and read again about as long as its bytes take at the unit's share of the memory rate, and
// add_cost is the second launch.  us with pieces of 16 at least and no add_cost / of 8 with it, both directions: 256 tokens at 8/2 heads 86.6 / 74.6
// (left whole), 389 tokens at 4/1 93.6 / 84.1, 2048 tokens at 4/1 160 / 143, a tick of 2048 query rows at 8/2 206 / 190.
inline void cut_where_worth(SchedGeom *g, const distca_ca_params *p, int32_t target, int32_t item_cost, int32_t piece_extra, int32_t add_cost) {
  const int32_t units = num_compute_units() / p->num_heads_kv;
  g->split_target = target;
  g->merge_tiles = 0;
  g->units_per_head = units > 0 ? units : 1;
  g->item_cost = item_cost;
  g->piece_extra = piece_extra;
  g->add_cost = add_cost;
  g->min_piece = kMinPieceWorth;
}
inline SchedGeom dq_geom(const distca_ca_params *p) {
  SchedGeom g = fwd_geom(p);
  g.rows_per_block = kDqRows;
  g.merge_tiles = merge_short_tasks(p) ? kMergeTilesDq : 0;  // in the list's cost unit, visible keys / kFwdKV
  return g;
}
inline SchedGeom bwd_geom(const distca_ca_params *p) {
  SchedGeom g;
  g.merge_tiles = 0;
  g.rows_per_block = kBwdRows;
  g.kv_per_block = kBwdKV;
  g.group = p->num_heads_q / p->num_heads_kv;
  g.causal = p->causal != 0;
  g.cost_shift = pick_cost_shift((int64_t)p->max_seqlen_q * g.group / kBwdRows + 1);
  g.split_target = bwd_split_target(p);
  g.min_piece = kMinPiece;
  g.units_per_head = g.item_cost = g.piece_extra = g.add_cost = 0;
  g.beside = 0.f;
  // one round of the dK/dV list per kv head: as many items as compute units serve that head (sched.h, kWalkUp)
  g.walk_round = num_compute_units() / p->num_heads_kv > 0 ? num_compute_units() / p->num_heads_kv : 1;
  return g;
}
// Whether a backward's lists share a launch.  preferred: the call brought that workspace (and may cut both lists).
inline int64_t dq_max_items(const distca_ca_params *p);
inline bool pair_backward(const distca_ca_params *p, bool preferred) {
  if (!few_row_blocks(p) || (int64_t)p->total_q * p->num_heads_q > (int64_t)kPairBlocksPerCU * kDqRows * num_compute_units()) return false;
  const int32_t target_kv = preferred ? preferred_key_pieces(p) : bwd_split_target(p);
  const int32_t target_q = preferred ? row_split_target(p, dq_max_items(p), kCutFromTilesDq) : 0;
  if (target_q == 0) return target_kv > 0 || few_key_blocks(p, kSplitFewPerCU);
  return target_kv > 0 && slots_apart(p, bwd_key_blocks_own_rows(p), target_kv, dq_max_items(p), target_q);
}
// Whether lists that share a launch are cut for the load of both.  Without a causal mask a task's blocks are all alike: cut as if alone, each list fills the units
// evenly, and sizes that follow from both lists leave an uneven end, which shows from some kCutForBothTiles tiles of the forward a unit on.  us backward, non-causal, cut for both /
// as if alone: 600 tokens at 32/8 heads (3 tiles) 51 / 73, 2048 at 4/1 (4) 77 / 88, 2048 at 8/2 (8) 98 / 101, 3000 at 4/1 (9) 101 / 108; 1000 at 64/8 (15) 138 / 131, 4096 at 4/1
// (16) 152 / 143, 3000 at 8/2 (17) 153 / 159, 4096 at 8/2 (32) 249 / 220, 8192 at 4/1 (64) 446 / 377 (one launch after the other 387), 4096 at 32/8 (128) 700 / 708.
constexpr int kCutForBothTiles = 12;
inline bool cut_for_both(const distca_ca_params *p) {
  return p->causal || (int64_t)p->total_q * p->num_heads_q * p->max_seqlen_k <= (int64_t)kCutForBothTiles * kFwdRows * kFwdKV * num_compute_units();
}
// Whether dQ's pieces are those of a list that shares its launch.  As row_split_target it must not know how K/V are stored (it once did: 8 tasks of 256 rows
// over a document of 16384 at 4/1 heads had 158 pieces over stored rows and 252 over copies, and dq other bits): it asks for the stored rows that one copy
// of every task's prefix would be, as far as the bounds tell, whole documents' (what row_tiles_to_gain takes for such) or the longest prefix for every task.
// Where it says no and the launch is shared all the same, pieces cut as if alone do as well or better.  us backward, 256 or 512 rows each, evenly over the
// prefixes, cut for both lists / as if alone: 8 tasks to 16384 at 4/1 heads 161 / 162, 16 to 16384 at 4/1 258 / 243, 8 to 16384 at 8/2 253 / 246, 2 to 4096
// at 32/8 142 / 128.
inline bool dq_pieces_beside(const distca_ca_params *p) {
  distca_ca_params q = *p;
  const int64_t copies = p->max_seqlen_q == p->max_seqlen_k && p->max_seqlen_k <= p->total_q ? p->total_q : (int64_t)p->max_seqlen_k * p->num_tasks;
  q.total_k = (int32_t)(copies < 0x7fffffff ? copies : 0x7fffffff);
  return pair_backward(&q, true);
}
// The lists as the calls launch them.  `target`: pieces aimed for per kv head, 0: whole blocks; for dK/dV also whether they are what
// the preferred workspace has room for (only what is worth it, at one size) or the smallest (equal parts).
inline SchedGeom launched_fwd_geom(const distca_ca_params *p, int32_t target) {
  SchedGeom g = launched_geom(fwd_geom(p), p);
  if (target > 0) cut_where_worth(&g, p, target, 6, 4, 8);
  return g;
}
inline SchedGeom launched_dq_geom(const distca_ca_params *p, int32_t target) {
  SchedGeom g = launched_geom(dq_geom(p), p);
  if (target > 0) {
    cut_where_worth(&g, p, target, 6, 3, 6);
    if (cut_for_both(p) && dq_pieces_beside(p)) g.beside = kDkdvBesideDq;
  }
  return g;
}
inline SchedGeom bwd_shared_geom(const distca_ca_params *p);
// beside: dQ's items share the launch (pair_backward)
inline SchedGeom launched_dkdv_geom(const distca_ca_params *p, int32_t target, bool preferred, bool shared, bool beside) {
  SchedGeom g = shared ? bwd_shared_geom(p) : bwd_geom(p);
  g.split_target = target;
  if (target > 0 && preferred) cut_where_worth(&g, p, target, 9, 14, 4);
  if (beside && cut_for_both(p)) g.beside = kDqBesideDkdv, g.min_piece = kMinPieceBeside;
  if (shared && target > 0) g.walk_round = 0;   // pieces count a group's visits downwards
  return g;
}
// Upper bound of the item count that needs only host-known sizes.
inline int64_t fwd_max_items(const distca_ca_params *p) {
  const int64_t group = p->num_heads_q / p->num_heads_kv;
  return (int64_t)p->total_q * group / kFwdRows + p->num_tasks + 1;
}
inline int64_t dq_max_items(const distca_ca_params *p) {
  const int64_t group = p->num_heads_q / p->num_heads_kv;
  return (int64_t)p->total_q * group / kDqRows + p->num_tasks + 1;
}
inline int64_t bwd_max_items(const distca_ca_params *p) {
  // Without cutting, items are (task, key block) over rows the task owns, or (group of tasks that share rows, key
  // block): either way the blocks tile stored rows.  With cutting (small batches only) tasks over shared rows have an
  // item per task and key block, and cutting adds at most total cost / piece <= split_target pieces (piece_size rounds up).
  return bwd_small_pieces(p) ? bwd_key_blocks_bound(p) + bwd_split_target(p) : bwd_key_blocks_own_rows(p);
}
// The dK/dV list over groups of tasks that share stored K/V rows: an item's cost is the sum over the group's tasks.
inline SchedGeom bwd_shared_geom(const distca_ca_params *p) {
  SchedGeom g = bwd_geom(p);
  g.split_target = 0;
  g.cost_shift = pick_cost_shift((int64_t)p->total_q * g.group / kBwdRows + p->num_tasks + 1);
  return g;
}

// One list to build: for a batch with these bounds, into region `ws`.
struct ListJob {
  const int32_t *cu_q, *cu_k;
  SchedGeom geom;
  int32_t *ws;
  int64_t max_items;
  SplitTables split;
};
// The dk / dv rows a backward clears: rows that no task reads.
struct BwdFill {
  uint8_t *dk, *dv;
  int64_t row_bytes;
  int32_t total_k;
  KvShards shards;
};
// The row statistics that the backward's kernels read, where a launch of their own makes them (attn_bwd_pair.hip): -<dO, O> and lse log2(e), [Hq][Tq].
struct RowStats {
  const uint8_t *dout, *out, *lse_tok;   // rows and lse as in BwdArgs
  const float *lse;
  const int64_t *task_off;
  int64_t tok_bytes;
  int32_t hq, total_q, f16;
  float *lse2, *neg_delta;               // null: no statistics
};
int launch_build_forward(const ListJob &j, int32_t num_tasks, hipStream_t stream);
// kv_off: null, or the tasks share stored K/V rows and the dK/dV list is made over groups of them (sched.h, SharedGroups; its region
// is sched_shared_region_bytes long)
int launch_build_backward(const ListJob &kv, const ListJob &q, const int32_t *kv_off, int32_t num_tasks, const BwdFill &fill, const RowStats &stats, hipStream_t stream);

inline int64_t align_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

}  // namespace distca
