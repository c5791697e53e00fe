// What the body of the dK/dV kernel (attn_bwd_dkdv64_kernel.inc) is written in; included inside a namespace, ahead of it.
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

// Adds up the pieces of the key blocks that were cut, in their order (cut_blocks.h, once for dK and once for dV: a workgroup has the keys
// of one half of one wave).  Bound by reading the slots (256 KB a piece).
__device__ __forceinline__ void add_up_dkdv(const BwdArgs &a, int part) {
  const int kvh = blockIdx.y, key_wave = (part >> 1) & 3, kb = part & 1, lane = threadIdx.x & 63, db = threadIdx.x >> 6;
  const int64_t kv_stride = (int64_t)a.hkv * kHeadDim;
  auto gradient = [&](bool is_dv) {
    add_up_cut_blocks(
        a.cut, a.slot,
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
  gradient(part >= kCutParts);
}
