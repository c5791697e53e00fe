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

constexpr int kThreads = 256;
constexpr int kBN = kBwdKV;    // keys per workgroup
constexpr int kBM = kBwdRows;  // flattened query rows per block
static_assert(kBN == 256 && kBM == 32, "tile geometry of this kernel");
constexpr int kRow = 256;      // bytes per tile row, chunks swizzled by tile_swz16
constexpr int kStages = 4;
constexpr int kTileQ = 0, kTileDO = kBM * kRow;
constexpr int kTileBytes = 2 * kBM * kRow;
constexpr int kStatBytes = 3 * kBM * 4;  // lse2, -delta, lim per row
constexpr int kStatOff = kStages * kTileBytes;
constexpr int kVOff = kStatOff + kStages * kStatBytes;
constexpr int kVWave = 64 * kRow + 64 * 16;  // a wave's resident V rows, in the tiles' layout, and (shards) where its rows go
// Of the four 32-element slices over d of a wave's V rows, as many as fit without spills inside the block loops stay in registers as
// B operands beside K; the rest is read from LDS every block.
constexpr int kVRegSlices = 3;
constexpr int kLds = kVOff + 4 * kVWave;
static_assert(kLds <= 160 * 1024, "LDS budget");
#ifndef DISTCA_RAWBAR
#define DISTCA_RAWBAR 1
#endif
constexpr int kLoadsPerBlock = 5;        // vector-memory instructions a wave issues per block
constexpr float kLog2e = 1.4426950408889634f;

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
// The lane's number, made where it is asked for (what the compiler knows how to make it makes once, and parks).
__device__ __forceinline__ int lane_now() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}
// This file is compiled with the compiler's default choice of MFMA form, which at 512 registers per wave keeps
// every MFMA result in the accumulation registers: right for the 256 dK / dV accumulators, which only MFMAs touch
// and which fill that file exactly.  The S and dP accumulators, which the vector ALU reads and overwrites, must
// live in the ordinary vector registers instead, and the only way to say so per instruction is to write those
// MFMAs as assembly with vector-register operands.  The compiler does not know what such a statement executes and
// so does not space its result from the vector instructions that read it (a four-pass MFMA: 8 wait states): the order of a block's
// instructions below, held in place by the scheduling fences, keeps at least three later MFMAs, each of which waits for the four passes
// of the one before it, between every such MFMA and the first read of its result, and spaced() does where a block's second half of keys
// is left out; a change to the block body has to keep that.
__device__ __forceinline__ void mfma16_v(f32x4 &acc, elemx8 a, elemx8 b) {
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_v0(f32x4 &acc, elemx8 a, elemx8 b) {  // acc = A B
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_vc(f32x4 &acc, elemx8 a, elemx8 b, const f32x4 &c0) {  // acc = A B + c0
  asm volatile(DISTCA_MFMA16_ASM " %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "v"(b), "v"(c0));
}

// First key, in the workgroup's block of 256, of a wave's first or second half of 32: the halves from the block's start go to waves
// 0, 1, 2, 3, 0, 1, 2, 3.  Every wave passes the same barrier per query block, so a block on the diagonal takes as long as the wave that
// sees most of it: with 64 keys in a row wave 0 has a whole block's work as soon as the first key is seen.  Dealt this way no wave has more
// than half a block's until the rows see 128 keys, nor ever where a task ends in a block of at most 128 keys.
// The kernel over 131072 tokens in documents of 64 / 128 / 256 / 512 / 2048, 32/8 heads, with 32x32x16 MFMAs, in us: 64 keys in a row 1526 / 1225 / 1168 /
// 1599 / 4426, in halves 1326 / 1115 / 1092 / 1536 / 4321 (a visit of half the work still takes 1.7 us of 2.0: requests, barrier and
// the chain from S to dK do not shrink with it).  (With the second halves in the order 3, 2, 1, 0 instead, wave 3's two lay side by side, and
// both could lie on the diagonal at once; now only one ever does, and only its elements are compared.)
__device__ __forceinline__ int dkdv_half_key(int wave, int half) { return kBN / 2 * half + 32 * wave; }

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

// Adds up the pieces of the key blocks that were cut, in their order (cut_blocks.h, once for dK and once for dV: a workgroup has the keys
// of one half of one wave).  Bound by reading the slots (256 KB a piece).
__global__ __launch_bounds__(kCutThreads) void ca_bwd_dkdv64_combine_kernel(BwdArgs a) {
  const int kvh = blockIdx.y, key_wave = (blockIdx.z >> 1) & 3, kb = blockIdx.z & 1, lane = threadIdx.x & 63, db = threadIdx.x >> 6;
  const int64_t kv_stride = (int64_t)a.hkv * kHeadDim;
  auto gradient = [&](bool is_dv) {
    add_up_cut_blocks(
        a.cut,
        [&](const int4 &e, f32x4 (&o)[4]) {
          const f32x4 *first = reinterpret_cast<const f32x4 *>(a.partial + ((int64_t)e.w * a.hkv + kvh) * kDkdvSlotBytes);
          add_pieces(first + ((is_dv ? 32 : 0) + 16 * kb + 4 * db) * kThreads + key_wave * 64 + lane, a.hkv * (kDkdvSlotBytes / 16), kThreads, e.z, o);
          if (!is_dv) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[k][r] *= a.scale;
          }
        },
        [&](const int4 &e, int r) -> elem_t * {
          const int ks = a.grp_off ? a.grp_off[e.x] : (a.kv_off ? a.kv_off[e.x] : a.cu_k[e.x]);
          const int kmax = a.grp_lmax ? a.grp_lmax[e.x] : a.cu_k[e.x + 1] - a.cu_k[e.x];
          const int key = e.y * kBN + dkdv_half_key(key_wave, kb) + r;
          if (key >= kmax) return nullptr;
          elem_t *out = is_dv ? a.dv : a.dk;
          int64_t row = ks + key;
          if (a.shards.num_shards > 0) {
            const int sh = find_shard(a.shards.row_start, a.shards.num_shards, ks + key);
            out += (is_dv ? a.shards.dv_off[sh] : a.shards.dk_off[sh]) / 2;
            row -= a.shards.row_start[sh];
          }
          return out + row * kv_stride + kvh * kHeadDim;
        });
  };
  gradient(blockIdx.z >= kCutParts);
}

}  // namespace

#ifndef DISTCA_F16
int dkdv64_lds_bytes() { return kLds; }
#endif

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
  if (max_cut > 0) hipLaunchKernelGGL(ca_bwd_dkdv64_combine_kernel, cut_grid(max_cut, a.hkv, 2 * kCutParts), dim3(kCutThreads), 0, stream, a);
  return DISTCA_OK;
}

}  // namespace distca
