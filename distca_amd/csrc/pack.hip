// fa2a shard pack / unpack and duplicate-gradient accumulation for gfx950.
//
// Behaviour follows the three kernels of the reference's csrc/core/memcpy.cu
// (memcpy_nvshmem_non_cp :22-74, memcpy_nvshmem_cp :77-155, inplace_grad_sum_kernel
// :158-236); the decomposition does not.  A shard is contiguous on both sides (rows
// start_s.. of the tensor, bytes offset_s.. of the buffer), so the job is a list of
// contiguous segment copies.  The logical token range is cut into one equal slice per
// workgroup; every wave locates the shard holding its slice's first token with a scan of
// the shard lengths in registers (no barrier), then the workgroup walks shards, streaming
// 16-byte vectors with non-temporal loads and stores (the data is touched once, keeping it
// out of L2 leaves the cache to whoever runs next).
//
// What a rank does around an all-to-all is several such copies at once, and each is a job of one
// launch (distca_exchange): q, k and v; a transport token made of several tensors' rows, put
// together or taken apart on the way instead of in a pass of its own; a row that goes to several
// replicas, read once; the rows of several replicas, or of several copies, added up on the way.
#include "api_util.h"
#include "common.h"

namespace distca {
namespace {

// What a plain 3 GiB device-to-device copy reaches on this part, by shape of the kernel (HBM peak 8 TB/s): 1024-thread
// workgroups over contiguous slices with 4 vectors per lane in flight 69.7 %, with 8 in flight 73 %; 512- and
// 256-thread workgroups 65-70 %; plain instead of non-temporal loads or stores 66-67 %; hipMemcpyDtoD 59 %.  Best is a
// workgroup that issues every load of its slice before its first store and then ends (one loop round per slice):
// 75-76 %; each further round of the same workgroup costs 2-4 %, and a slice that ends in a round of fewer vectors
// loses more (16 in flight over a slice of one and a half rounds: 68 %).  So a slice is one round where tokens
// allow, and the last, partial round of a run inside a shard is issued like a whole one with the lanes past the end
// switched off.  On the 262 144-token q/k/v workload, one launch for the three tensors: 10 vectors per lane
// (160 KiB slices) 75.4 / 75.3 % packing / unpacking, 16 (256 KiB) 75.0 / 75.5 %, 8 in three rounds 70.7 / 71.7 %,
// 20 or 24 in one round 73 %, 32 in one round 65 %.
constexpr int kPackThreads = 1024;
#ifndef DISTCA_PACK_UNROLL
#define DISTCA_PACK_UNROLL 10
#endif
constexpr int kUnroll = DISTCA_PACK_UNROLL;
constexpr int64_t kVecRound = (int64_t)kPackThreads * 16;      // bytes of one vector per thread
constexpr int64_t kRoundBytes = kUnroll * kVecRound;           // bytes a workgroup moves per loop round
// Tokens of several parts compute an address per vector: eight in flight keep to the 64 registers of two workgroups per unit.
constexpr int kUnrollParts = 8;
// Jobs that add rows up hold fp32 sums beside the loads: six vectors per lane in flight (of two-byte elements: 48 + 24 registers)
constexpr int kUnrollSum = 6;

// The shard that holds position `pos` of the concatenated shard list (idx == num_seq: none) and the position of its first
// token.  Every wave finds it for itself: four loads of 64 lengths at a time, a scan over the lanes, no barrier.  (A block-wide
// scan did this before: with its barriers 2 to 3 us of a small copy's 7.)
struct Segment {
  int idx;
  int64_t start;
};
__device__ __forceinline__ int64_t lane_value(int64_t v, int lane) {
  const uint64_t u = (uint64_t)v;
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), lane), lo = (uint32_t)__builtin_amdgcn_readlane((int)u, lane);
  return (int64_t)((hi << 32) | lo);
}
__device__ __forceinline__ Segment find_segment(const int64_t *__restrict__ seq_tokens, int num_seq, int64_t pos) {
  constexpr int kAhead = 4;
  const int lane = threadIdx.x & 63;
  int64_t before = 0;
  for (int c0 = 0; c0 < num_seq; c0 += 64 * kAhead) {
    int64_t len[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int i = c0 + 64 * j + lane;
      len[j] = i < num_seq ? seq_tokens[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      int64_t incl = len[j];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int64_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      const unsigned long long past = __ballot(before + incl > pos);
      if (past) {
        const int l = __builtin_ctzll(past);
        return Segment{c0 + 64 * j + l, before + lane_value(incl, l) - lane_value(len[j], l)};
      }
      before += lane_value(incl, 63);
    }
  }
  return Segment{num_seq, 0};
}

// One copy: `part_vecs` vectors of every token, at `pitch` bytes in the tensor and from vector `part_v0` of the token on in the
// buffer.  (The parts of a token are jobs of their own.)
struct Job {
  uint8_t *data;   // null: the bytes are zeros (the padding of a token)
  const int64_t *seq_offset, *seq_tokens;
  const int8_t *mask;
  const int32_t *num_copies;
  const int64_t *copy_start;
  int64_t num_tokens, token_bytes, pitch;
  int32_t kind, dtype, num_seq, max_cp, max_copies, tokens_per_wg, first_wg;
  uint32_t part_v0, part_vecs, magic;  // magic = ceil(2^32 / part_vecs) (0: part_vecs is 1): i / part_vecs == umulhi(i, magic) for i * part_vecs < 2^32
  __host__ __device__ bool whole() const { return pitch == token_bytes && (int64_t)part_vecs * 16 == token_bytes; }
};
constexpr int kMaxJobs = 12;
struct Jobs {
  Job job[kMaxJobs];
  int32_t n;
};

// (Each job's first workgroup lies with its other fields: the look at all of them brings those along.  Beside each other they are one trip to memory, and the
// job's fields a second one: 0.6 us of a launch.)
__device__ __forceinline__ int job_of_workgroup(const Jobs &jobs) {
  int j = 0;
#pragma unroll
  for (int i = 1; i < kMaxJobs; ++i)
    if (i < jobs.n && (int)blockIdx.x >= jobs.job[i].first_wg) j = i;
  return j;
}

// A contiguous run of memory as a buffer resource of its exact length: lanes past its end load zeros and store nothing, so a
// partial round needs no branches and is issued like a whole one.  (With a predicate per vector the compiler could not keep
// the loop in the 64 registers that let two workgroups share a compute unit.)
typedef __amdgpu_buffer_rsrc_t run_t;
__device__ __forceinline__ run_t make_run(const void *p, uint32_t nvec) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(uniform_ptr(p)), 0, uniform_int((int)(nvec << 4)), 0x00020000);
}
constexpr int kNonTemporal = 2;
constexpr int kNowhere = (int)0x80000000u;   // an offset past the end of every run
__device__ __forceinline__ u32x4 load_nt(run_t r, int i) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, i << 4, 0, kNonTemporal)); }
__device__ __forceinline__ void store_nt(run_t r, int i, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, r, i << 4, 0, kNonTemporal); }
__device__ __forceinline__ u32x4 load_at(run_t r, uint32_t byte, bool ok) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, ok ? (int)byte : kNowhere, 0, kNonTemporal));
}
__device__ __forceinline__ void store_at(run_t r, uint32_t byte, bool ok, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, r, ok ? (int)byte : kNowhere, 0, kNonTemporal); }
// N vectors per lane at a time, all loads of a round issued before its first store.
template <int N, class Load, class Use>
__device__ __forceinline__ void rounds(uint32_t nvec, Load load, Use use) {
  for (int i = threadIdx.x; i < (int)nvec; i += N * kPackThreads) {
    u32x4 r[N];
#pragma unroll
    for (int u = 0; u < N; ++u) r[u] = load(i + u * kPackThreads);
    int j = i;   // (opaque: what the second half derives from it is computed there, not kept in registers across the loads)
    asm volatile("" : "+v"(j));
#pragma unroll
    for (int u = 0; u < N; ++u) use(j + u * kPackThreads, r[u]);
  }
}
__device__ __forceinline__ void copy_run(uint8_t *dst, const uint8_t *src, uint32_t nvec) {
  const run_t d = make_run(dst, nvec), s = make_run(src, nvec);
  rounds<kUnroll>(nvec, [&](int i) { return load_nt(s, i); }, [&](int i, u32x4 v) { store_nt(d, i, v); });
}

// `n` tokens of a job that covers a part of each, from row `row` on, at `buf` in the buffer: both sides are rows at a pitch.
template <bool TO_BUF>
__device__ __forceinline__ void copy_part(const Job &jb, uint8_t *buf, int64_t row, uint32_t n) {
  const uint32_t nvec = n * jb.part_vecs;
  const uint32_t tp = (uint32_t)jb.pitch, bp = (uint32_t)jb.token_bytes;
  const uint32_t last = jb.part_vecs;   // the run of a side ends with the part of its last token
  const run_t ten = make_run(jb.data + row * jb.pitch, jb.data ? (n - 1) * (tp >> 4) + last : 0);
  const run_t b = make_run(buf + (int64_t)jb.part_v0 * 16, (n - 1) * (bp >> 4) + last);
  auto token_of = [&](int i) { return jb.magic ? __umulhi((uint32_t)i, jb.magic) : (uint32_t)i; };
  rounds<kUnrollParts>(nvec,
                       [&](int i) {
                         const uint32_t t = token_of(i), c = i - t * jb.part_vecs;
                         return load_at(TO_BUF ? ten : b, t * (TO_BUF ? tp : bp) + (c << 4), i < (int)nvec);
                       },
                       [&](int i, u32x4 v) {
                         const uint32_t t = token_of(i), c = i - t * jb.part_vecs;
                         store_at(TO_BUF ? b : ten, t * (TO_BUF ? bp : tp) + (c << 4), i < (int)nvec, v);
                       });
}

template <typename T>
struct Add;
template <>
struct Add<float> {
  static __device__ __forceinline__ u32x4 apply(u32x4 a, u32x4 b) {
    f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
    f32x4 r = {x[0] + y[0], x[1] + y[1], x[2] + y[2], x[3] + y[3]};
    return __builtin_bit_cast(u32x4, r);
  }
};
template <>
struct Add<_Float16> {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ u32x4 apply(u32x4 a, u32x4 b) {
    h8 x = __builtin_bit_cast(h8, a), y = __builtin_bit_cast(h8, b);
    h8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = x[i] + y[i];
    return __builtin_bit_cast(u32x4, r);
  }
};
template <>
struct Add<__bf16> {
  // bf16 + bf16: exact in fp32 up to one rounding that never lands on a bf16 tie, so
  // fp32 add followed by round-to-nearest-even equals the correctly rounded bf16 sum.
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ u32x4 apply(u32x4 a, u32x4 b) {
    bf16x8 x = __builtin_bit_cast(bf16x8, a), y = __builtin_bit_cast(bf16x8, b);
    f32x8 fx = __builtin_convertvector(x, f32x8), fy = __builtin_convertvector(y, f32x8);
    f32x8 s;
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = fx[i] + fy[i];
    return __builtin_bit_cast(u32x4, __builtin_convertvector(s, bf16x8));
  }
};


// Sums in fp32 of the rows of several replicas, rounded once.
template <typename T>
struct Sum {
  static constexpr int kN = 16 / sizeof(T);
  float s[kN];
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  typedef float fvec __attribute__((ext_vector_type(16 / sizeof(T))));
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < kN; ++i) s[i] = 0.f;
  }
  __device__ __forceinline__ void add(u32x4 v) {
    const fvec f = __builtin_convertvector(__builtin_bit_cast(vec, v), fvec);
#pragma unroll
    for (int i = 0; i < kN; ++i) s[i] += f[i];
  }
  __device__ __forceinline__ u32x4 value() const {
    fvec f;
#pragma unroll
    for (int i = 0; i < kN; ++i) f[i] = s[i];
    return __builtin_bit_cast(u32x4, __builtin_convertvector(f, vec));
  }
};
template <typename T>
__device__ __forceinline__ void sum_replicas(const Job &jb, const uint8_t *buffer, int seg, int64_t skip, uint8_t *dst_p, uint32_t nvec) {
  const run_t dst = make_run(dst_p, nvec);
  for (int i = threadIdx.x; i < (int)nvec; i += kUnrollSum * kPackThreads) {
    Sum<T> acc[kUnrollSum];
#pragma unroll
    for (int u = 0; u < kUnrollSum; ++u) acc[u].clear();
    for (int c = 0; c < jb.max_cp; ++c) {
      if (!uniform_int(jb.mask[(int64_t)seg * jb.max_cp + c])) continue;
      const run_t src = make_run(buffer + jb.seq_offset[(int64_t)c * jb.num_seq + seg] + skip, nvec);
      u32x4 r[kUnrollSum];
#pragma unroll
      for (int u = 0; u < kUnrollSum; ++u) r[u] = load_nt(src, i + u * kPackThreads);
#pragma unroll
      for (int u = 0; u < kUnrollSum; ++u) acc[u].add(r[u]);
    }
#pragma unroll
    for (int u = 0; u < kUnrollSum; ++u) store_nt(dst, i + u * kPackThreads, acc[u].value());
  }
}
// Rows of a main copy: the rows of its copies added in order, one rounding per addition; the sum stays in the tensor
// and, when the shard is sent (buf not null), goes to the buffer.
template <typename T>
__device__ __forceinline__ void sum_copies(const Job &jb, int seg, int64_t skip_rows, int32_t nc, uint8_t *main_p, uint8_t *buf, uint32_t nvec) {
  const int64_t *starts = jb.copy_start + (int64_t)seg * jb.max_copies;
  const run_t rows = make_run(main_p, nvec), sent = make_run(buf, buf ? nvec : 0);
  for (int i = threadIdx.x; i < (int)nvec; i += kUnrollSum * kPackThreads) {
    u32x4 m[kUnrollSum];
#pragma unroll
    for (int u = 0; u < kUnrollSum; ++u) m[u] = load_nt(rows, i + u * kPackThreads);
    for (int32_t c = 0; c < nc; ++c) {
      const run_t src = make_run(jb.data + (starts[c] + skip_rows) * jb.token_bytes, nvec);
      u32x4 r[kUnrollSum];
#pragma unroll
      for (int u = 0; u < kUnrollSum; ++u) r[u] = load_nt(src, i + u * kPackThreads);
#pragma unroll
      for (int u = 0; u < kUnrollSum; ++u) m[u] = Add<T>::apply(m[u], r[u]);
    }
#pragma unroll
    for (int u = 0; u < kUnrollSum; ++u) {
      store_nt(rows, i + u * kPackThreads, m[u]);
      store_nt(sent, i + u * kPackThreads, m[u]);
    }
  }
}

// The jobs of one call: workgroups [first_wg, first_wg of the next job) serve a job, each a slice of its tokens.  One
// launch has one tail instead of one per tensor, and the small tensors' slices fill the gaps the large one leaves.
// PARTS: with jobs whose tokens have several parts; SUMS: with jobs that add rows up.  Launches without either are spared their
// registers, so that two workgroups fit a compute unit.
template <bool TO_BUF, bool PARTS, bool SUMS>
__global__ __launch_bounds__(kPackThreads, SUMS ? 4 : 8) void exchange_kernel(Jobs jobs, uint8_t *buffer) {
  const int j = job_of_workgroup(jobs);
  const Job &jb = jobs.job[j];
  const int64_t t0 = (int64_t)((int)blockIdx.x - jb.first_wg) * jb.tokens_per_wg;
  int64_t t1 = t0 + jb.tokens_per_wg;
  if (t1 > jb.num_tokens) t1 = jb.num_tokens;
  if (t0 >= t1) return;
  Segment sg = find_segment(jb.seq_tokens, jb.num_seq, t0);
  int seg = sg.idx;
  int64_t seg_start = seg < jb.num_seq ? sg.start : t0;
  const int64_t tb = jb.token_bytes;
  const bool replicas = jb.kind == DISTCA_JOB_REPLICAS || jb.kind == DISTCA_JOB_REPLICA_SUM;
  for (; seg < jb.num_seq && seg_start < t1; ++seg) {
    const int64_t seg_end = seg_start + uniform_int64(jb.seq_tokens[seg]);
    const int64_t a = seg_start > t0 ? seg_start : t0, b = seg_end < t1 ? seg_end : t1;
    const int64_t skip = (a - seg_start) * tb;
    seg_start = seg_end;
    if (a >= b) continue;
    const uint32_t nvec = (uint32_t)((b - a) * (tb >> 4));
    if (replicas) {
      if (SUMS && jb.kind == DISTCA_JOB_REPLICA_SUM) {
        uint8_t *dst = jb.data + a * tb;
        if (jb.dtype == DISTCA_DTYPE_BF16) sum_replicas<__bf16>(jb, buffer, seg, skip, dst, nvec);
        else if (jb.dtype == DISTCA_DTYPE_F16) sum_replicas<_Float16>(jb, buffer, seg, skip, dst, nvec);
        else sum_replicas<float>(jb, buffer, seg, skip, dst, nvec);
        continue;
      }
      if (TO_BUF) {
        // every live replica gets the rows, which are read once
        const run_t src = make_run(jb.data + a * tb, nvec);
        for (int i = threadIdx.x; i < (int)nvec; i += kUnroll * kPackThreads) {
          u32x4 r[kUnroll];
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) r[u] = load_nt(src, i + u * kPackThreads);
          for (int c = 0; c < jb.max_cp; ++c) {
            if (!uniform_int(jb.mask[(int64_t)seg * jb.max_cp + c])) continue;
            const run_t dst = make_run(buffer + jb.seq_offset[(int64_t)c * jb.num_seq + seg] + skip, nvec);
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) store_nt(dst, i + u * kPackThreads, r[u]);
          }
        }
      } else {
        for (int c = 0; c < jb.max_cp; ++c) {
          if (!uniform_int(jb.mask[(int64_t)seg * jb.max_cp + c])) continue;
          copy_run(jb.data + (c * jb.num_tokens + a) * tb, buffer + jb.seq_offset[(int64_t)c * jb.num_seq + seg] + skip, nvec);
        }
      }
      continue;
    }
    const bool sent = !TO_BUF || !jb.mask || uniform_int(jb.mask[seg]) != 0;
    uint8_t *buf = buffer + (sent ? jb.seq_offset[seg] + skip : 0);
    if (SUMS && jb.kind == DISTCA_JOB_COPY_SUM) {
      const int32_t nc = uniform_int(jb.num_copies[seg]);
      if (nc > 0) {
        uint8_t *m = jb.data + a * tb, *dst = sent ? buf : nullptr;
        if (jb.dtype == DISTCA_DTYPE_BF16) sum_copies<__bf16>(jb, seg, skip / tb, nc, m, dst, nvec);
        else if (jb.dtype == DISTCA_DTYPE_F16) sum_copies<_Float16>(jb, seg, skip / tb, nc, m, dst, nvec);
        else sum_copies<float>(jb, seg, skip / tb, nc, m, dst, nvec);
        continue;
      }
    }
    if (!sent) continue;
    if (PARTS && !jb.whole()) {
      copy_part<TO_BUF>(jb, buf, a, (uint32_t)(b - a));
      continue;
    }
    uint8_t *ten = jb.data + a * tb;
    if (TO_BUF) copy_run(buf, ten, nvec);
    else copy_run(ten, buf, nvec);
  }
  if (SUMS && jb.kind == DISTCA_JOB_REPLICA_SUM && seg_start < t1) {   // rows behind the last shard: sums of nothing
    const uint32_t nvec = (uint32_t)((t1 - seg_start) * (tb >> 4));
    const run_t dst = make_run(jb.data + seg_start * tb, nvec);
    for (int i = threadIdx.x; i < (int)nvec; i += kPackThreads) store_nt(dst, i, u32x4{0, 0, 0, 0});
  }
}

// ---- Up to some 30 to 130 MB: a vector a thread ----
//
// A launch of a few MB is a chain of trips to memory, not a matter of bandwidth: a plain copy of 3 MB takes 2.4 us, and the same by
// exchange_kernel took 6 to 8, because a slice's runs go one after the other (a trip there and a trip back for each shard and replica it
// touches), behind a shard's length, place and mask and the replicas' masks and places read one by one.  Here a thread moves one vector,
// whatever shard it lies in: a wave reads the lengths, places and masks of 64 shards at once, a lane a shard, finds by lane moves where its
// vectors go, and all of them travel together; what is packed is requested before the list is read.
// us by slices / by vectors, pack, reply, request and gradients of the linear side: 1024 tokens at 8/2 heads (3 / 2 / 7 / 3 MB)
// 7.7 7.1 11.5 9.0 / 4.3 3.9 6.0 5.0.  Which of the two a launch takes: vectors_gain.
constexpr int kVectorThreads = 256;
constexpr int kVectorSeqs = 256;             // shards of a job: four reads of 64

// 64 shards from c0 on, one a lane.  end: position behind the shard's last token (sums saturate; tensors have fewer than 2^31 tokens).
struct ShardWindow {
  uint32_t len, end;
  int64_t off;
  int sent;
};
__device__ __forceinline__ uint32_t add_tokens(uint32_t a, uint32_t b) { return __builtin_elementwise_add_sat(a, b); }
__device__ __forceinline__ ShardWindow read_shards(const Job &jb, bool plain, const int8_t *mask, int c0, uint32_t before) {
  const int i = c0 + (threadIdx.x & 63);
  ShardWindow w{0, 0, 0, 1};
  if (i < jb.num_seq) {
    const int64_t n = jb.seq_tokens[i];
    if (plain) w.off = jb.seq_offset[i];
    if (mask) w.sent = mask[i];
    w.len = n <= 0 ? 0u : (n > 0x7fffffff ? 0x7fffffffu : (uint32_t)n);
  }
  uint32_t v = w.len;   // inclusive sums over the lanes, by DPP moves
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1 and 3
  v = add_tokens(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2 and 3
  w.end = add_tokens(before, v);
  return w;
}
__device__ __forceinline__ u32x4 load_vec(const uint8_t *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ void store_vec(uint8_t *p, u32x4 v) { *reinterpret_cast<u32x4 *>(p) = v; }

// f(replica, its place) for every live replica of shard `seg`, in their order: masks and places are read a lane a replica.  By whole waves.
template <class F>
__device__ __forceinline__ void each_replica(const Job &jb, int seg, F f) {
  for (int c0 = 0; c0 < jb.max_cp; c0 += 64) {
    const int c = c0 + (threadIdx.x & 63);
    int on = 0;
    int64_t off = 0;
    if (c < jb.max_cp) {
      on = jb.mask[(int64_t)seg * jb.max_cp + c];
      off = jb.seq_offset[(int64_t)c * jb.num_seq + seg];
    }
    for (unsigned long long m = __ballot(on != 0); m; m &= m - 1) f(c0 + __builtin_ctzll(m), lane_value(off, __builtin_ctzll(m)));
  }
}
// f(first row of the copy) for the copies of shard `seg`, in their order.  By whole waves.
template <class F>
__device__ __forceinline__ int each_copy(const Job &jb, int seg, F f) {
  const int64_t *starts = jb.copy_start + (int64_t)seg * jb.max_copies;
  const int lane = threadIdx.x & 63;
  const int32_t given = jb.num_copies[seg];
  int64_t start = lane < jb.max_copies ? starts[lane] : 0;
  const int32_t nc = uniform_int(given);
  for (int c = 0; c < nc; ++c) {
    if (c > 0 && (c & 63) == 0) start = c + lane < jb.max_copies ? starts[c + lane] : 0;
    f(lane_value(start, c & 63));
  }
  return nc;
}

template <bool TO_BUF, typename T>
__device__ __forceinline__ void vector_sum(const Job &jb, uint8_t *buffer, int seg, const ShardWindow &w, int l, uint32_t row, bool in, uint32_t byte, uint8_t *at) {
  if (!TO_BUF) {
    Sum<T> acc;
    acc.clear();
    each_replica(jb, seg, [&](int, int64_t off) {
      if (in) acc.add(load_vec(buffer + off + (int64_t)row * jb.token_bytes + byte));
    });
    if (in) store_vec(at, acc.value());
    return;
  }
  u32x4 m = u32x4{0, 0, 0, 0};
  if (in) m = load_vec(at);
  const int nc = each_copy(jb, seg, [&](int64_t start) {
    if (in) m = Add<T>::apply(m, load_vec(jb.data + (start + row) * jb.token_bytes + byte));
  });
  const int64_t off = lane_value(w.off, l);
  const bool sent = __builtin_amdgcn_readlane(w.sent, l) != 0;
  if (in && nc > 0) store_vec(at, m);
  if (in && sent) store_vec(buffer + off + (int64_t)row * jb.token_bytes + byte, m);
}

template <bool TO_BUF>
__global__ __launch_bounds__(kVectorThreads) void exchange_vectors_kernel(Jobs jobs, uint8_t *buffer) {
  const int j = job_of_workgroup(jobs);
  const Job &jb = jobs.job[j];
  const int lane = threadIdx.x & 63;
  const uint32_t nvec = (uint32_t)jb.num_tokens * jb.part_vecs, i = (uint32_t)((int)blockIdx.x - jb.first_wg) * kVectorThreads + threadIdx.x;
  const uint32_t first = (uint32_t)uniform_int((int)(i - lane));
  if (first >= nvec) return;
  const bool live = i < nvec;
  const uint32_t ic = live ? i : nvec - 1;
  const uint32_t t = jb.magic ? __umulhi(ic, jb.magic) : ic, byte = (ic - t * jb.part_vecs) << 4;   // token, and place in its part
  const uint32_t t_first = (uint32_t)uniform_int((int)t), t_last = (uint32_t)__builtin_amdgcn_readlane((int)t, 63);
  uint8_t *at = jb.data + (int64_t)t * jb.pitch + byte;
  const int kind = jb.kind;
  const bool plain = kind == DISTCA_JOB_PLAIN, sums = kind == DISTCA_JOB_REPLICA_SUM || kind == DISTCA_JOB_COPY_SUM;
  const bool by_shard = plain || kind == DISTCA_JOB_COPY_SUM;   // (else by shard and replica)
  u32x4 v = u32x4{0, 0, 0, 0};
  if (TO_BUF && !sums && live && jb.data) v = load_vec(at);

  // the shard of the wave's first token
  const int8_t *mask = TO_BUF && by_shard ? jb.mask : nullptr;
  int c0 = 0, seg = jb.num_seq;
  ShardWindow w{0, 0, 0, 0};
  uint32_t before = 0;
  for (; c0 < jb.num_seq; c0 += 64) {
    w = read_shards(jb, by_shard, mask, c0, before);
    const unsigned long long past = __ballot(w.end > t_first);
    if (past) {
      seg = c0 + __builtin_ctzll(past);
      break;
    }
    before = (uint32_t)__builtin_amdgcn_readlane((int)w.end, 63);
  }
  // and, from there on, those of all of its tokens
  bool found = false;   // this vector has a place
  uint8_t *place = buffer;
  for (; seg < jb.num_seq; ++seg) {
    if (seg - c0 == 64) {
      before = (uint32_t)__builtin_amdgcn_readlane((int)w.end, 63);
      c0 += 64;
      w = read_shards(jb, by_shard, mask, c0, before);
    }
    const int l = seg - c0;
    const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)w.end, l), start = end - (uint32_t)__builtin_amdgcn_readlane((int)w.len, l);
    if (start > t_last) break;
    const bool in = live && t >= start && t < end;
    const uint32_t row = t - start;   // (of the shard, where `in`)
    if (plain) {
      if (in && __builtin_amdgcn_readlane(w.sent, l) != 0) {
        found = true;
        place = buffer + lane_value(w.off, l) + (int64_t)row * jb.token_bytes + (((int64_t)jb.part_v0 << 4) + byte);
      }
    } else if (sums) {
      found = found || in;
      if (jb.dtype == DISTCA_DTYPE_BF16) vector_sum<TO_BUF, __bf16>(jb, buffer, seg, w, l, row, in, byte, at);
      else if (jb.dtype == DISTCA_DTYPE_F16) vector_sum<TO_BUF, _Float16>(jb, buffer, seg, w, l, row, in, byte, at);
      else vector_sum<TO_BUF, float>(jb, buffer, seg, w, l, row, in, byte, at);
    } else {
      each_replica(jb, seg, [&](int c, int64_t off) {
        uint8_t *b = buffer + off + (int64_t)row * jb.token_bytes + byte;
        if (!in) return;
        if (TO_BUF) store_vec(b, v);
        else store_vec(at + (int64_t)c * jb.num_tokens * jb.token_bytes, load_vec(b));
      });
    }
  }
  if (plain && found) {
    if (TO_BUF) store_vec(place, v);
    else store_vec(at, load_vec(place));
  }
  if (!TO_BUF && kind == DISTCA_JOB_REPLICA_SUM && live && !found) store_vec(at, v);   // rows behind the last shard: sums of nothing
}

// data[start_s + t] += data[copy_start_id[s][c] + t] for c = 0..num_copies[s]-1 in order,
// one rounding per addition.  Rows are cut into per-workgroup slices like those of exchange_kernel.
template <typename T>
__global__ __launch_bounds__(kPackThreads) void grad_sum_kernel(T *__restrict__ data, const int32_t *__restrict__ num_copies,
                                                              const int64_t *__restrict__ copy_start_id,
                                                              const int64_t *__restrict__ seq_lens, int64_t num_tokens,
                                                              int64_t hidden, int64_t num_seq, int64_t max_copies,
                                                              int64_t tokens_per_wg) {
  int64_t t0 = (int64_t)blockIdx.x * tokens_per_wg;
  int64_t t1 = t0 + tokens_per_wg;
  if (t1 > num_tokens) t1 = num_tokens;
  if (t0 >= t1) return;
  const Segment sg = find_segment(seq_lens, (int)num_seq, t0);
  if (sg.idx >= num_seq) return;
  int64_t seg = sg.idx, seg_start = sg.start;
  constexpr int kPerVec = 16 / sizeof(T);
  const int64_t row_vecs = hidden / kPerVec;        // vector part of a row
  const int64_t row_tail = hidden - row_vecs * kPerVec;
  while (seg_start < t1 && seg < num_seq) {
    const int64_t len = seq_lens[seg];
    const int64_t seg_end = seg_start + len;
    const int32_t nc = num_copies[seg];
    const int64_t a = seg_start > t0 ? seg_start : t0;
    const int64_t b = seg_end < t1 ? seg_end : t1;
    if (nc > 0 && a < b) {
      const int64_t *starts = copy_start_id + seg * max_copies;
      if (row_tail == 0 && ((hidden * sizeof(T)) & 15) == 0) {
        // rows are whole 16-byte vectors and contiguous: treat [a,b) as one vector run
        const int64_t nvec = (b - a) * row_vecs;
        u32x4 *main_p = reinterpret_cast<u32x4 *>(data + a * hidden);
        for (int64_t i = threadIdx.x; i < nvec; i += kPackThreads) {
          u32x4 m = main_p[i];
          for (int32_t c = 0; c < nc; ++c) {
            const u32x4 *cp = reinterpret_cast<const u32x4 *>(data + (starts[c] + (a - seg_start)) * hidden);
            m = Add<T>::apply(m, __builtin_nontemporal_load(cp + i));
          }
          main_p[i] = m;
        }
      } else {
        const int64_t n = (b - a) * hidden;
        T *main_p = data + a * hidden;
        for (int64_t i = threadIdx.x; i < n; i += kPackThreads) {
          T m = main_p[i];
          for (int32_t c = 0; c < nc; ++c) m = (T)(m + data[(starts[c] + (a - seg_start)) * hidden + i]);
          main_p[i] = m;
        }
      }
    }
    seg_start = seg_end;
    ++seg;
  }
}

// Bytes of a workgroup's slice for a launch of `total` bytes: one loop round (160 KiB at 10 vectors per lane) once the launch
// has four such slices per compute unit; below that as many whole vectors per thread as give every unit two workgroups, so
// that a small copy (of more shards than exchange_vectors_kernel takes) is spread over the device.
int64_t slice_bytes(int64_t total) {
  const int64_t cus = num_compute_units();
  if (total >= 4 * cus * kRoundBytes) return kRoundBytes;
  int64_t b = (total / (2 * cus) + kVecRound - 1) / kVecRound * kVecRound;
  return b < kVecRound ? kVecRound : (b > kRoundBytes ? kRoundBytes : b);
}
int64_t slice_tokens(int64_t slice, int64_t tokens, int64_t token_bytes, int64_t *grid) {
  int64_t per = (slice + token_bytes / 2) / token_bytes;
  if (per < 1) per = 1;
  *grid = (tokens + per - 1) / per;
  return per;
}

// Checks one job and appends it; 0 when it was empty.
int add_job(Jobs *jobs, const distca_exchange_job &in, int64_t token_bytes, int to_buffer, const void *buffer, const char *what) {
  const bool replicas = in.kind == DISTCA_JOB_REPLICAS || in.kind == DISTCA_JOB_REPLICA_SUM;
  if (in.num_seq < 0 || in.num_tokens < 0 || token_bytes < 0 || (replicas && in.max_cp < 0)) return fail(DISTCA_E_INVALID, "%s: negative size", what);
  // (a sum over replicas writes its rows also where there is no shard or no replica: as zeros, and nothing else of the job is read)
  const int64_t num_seq = replicas && in.max_cp == 0 ? 0 : in.num_seq;
  if (in.num_tokens == 0 || token_bytes == 0 || (num_seq == 0 && in.kind != DISTCA_JOB_REPLICA_SUM)) return 0;
  if (num_seq > 0 && (!buffer || !in.seq_offset || !in.seq_tokens || (replicas && !in.mask))) return fail(DISTCA_E_INVALID, "%s: null pointer", what);
  if (token_bytes % 16) return fail(DISTCA_E_INVALID, "%s: token_bytes=%lld is not a multiple of 16", what, (long long)token_bytes);
  if (in.num_tokens * (replicas && in.max_cp > 0 ? in.max_cp : 1) >= (1ll << 31) || in.num_seq >= (1ll << 31) || token_bytes >= (1ll << 31))
    return fail(DISTCA_E_INVALID, "%s: num_tokens%s must be < 2^31", what, replicas ? "*max_cp" : "");
  if (in.kind == DISTCA_JOB_REPLICA_SUM && to_buffer) return fail(DISTCA_E_INVALID, "%s: a sum over replicas only unpacks", what);
  if (in.kind == DISTCA_JOB_COPY_SUM && !to_buffer) return fail(DISTCA_E_INVALID, "%s: a sum over copies only packs", what);
  if (in.kind == DISTCA_JOB_REPLICA_SUM || in.kind == DISTCA_JOB_COPY_SUM) {
    if (in.dtype != DISTCA_DTYPE_F32 && in.dtype != DISTCA_DTYPE_F16 && in.dtype != DISTCA_DTYPE_BF16)
      return fail(DISTCA_E_UNSUPPORTED, "%s: dtype %lld (only fp32, fp16, bf16)", what, (long long)in.dtype);
    if (in.kind == DISTCA_JOB_COPY_SUM && in.max_copies < 0) return fail(DISTCA_E_INVALID, "%s: negative size", what);
    if (in.kind == DISTCA_JOB_COPY_SUM && in.max_copies > 0 && (!in.num_copies || !in.copy_start)) return fail(DISTCA_E_INVALID, "%s: null pointer", what);
  }
  const int64_t kind = in.kind == DISTCA_JOB_COPY_SUM && in.max_copies == 0 ? DISTCA_JOB_PLAIN : in.kind;   // no copies to add up
  const bool whole = in.num_parts == 1 && in.part[0].bytes == token_bytes && in.part[0].pitch == token_bytes;
  if (!whole && in.kind != DISTCA_JOB_PLAIN) return fail(DISTCA_E_INVALID, "%s: replicas and sums take whole tokens", what);
  if (!whole && token_bytes > (1 << 19)) return fail(DISTCA_E_UNSUPPORTED, "%s: tokens of several parts hold at most 512 KiB", what);
  int64_t at = 0;
  auto append = [&](void *data, int64_t pitch, int64_t bytes) {
    if (jobs->n == kMaxJobs) return fail(DISTCA_E_INVALID, "%s: more than %d parts in one launch", what, kMaxJobs);
    Job &o = jobs->job[jobs->n++];
    o.data = (uint8_t *)data;
    o.seq_offset = in.seq_offset; o.seq_tokens = in.seq_tokens; o.mask = in.mask;
    o.num_copies = in.num_copies; o.copy_start = in.copy_start;
    o.num_tokens = in.num_tokens; o.token_bytes = token_bytes; o.pitch = pitch;
    o.kind = (int32_t)kind; o.dtype = (int32_t)in.dtype;
    o.num_seq = (int32_t)num_seq; o.max_cp = (int32_t)in.max_cp; o.max_copies = (int32_t)in.max_copies;
    o.part_v0 = (uint32_t)(at / 16); o.part_vecs = (uint32_t)(bytes / 16);
    o.magic = o.part_vecs == 1 ? 0u : (uint32_t)(((1ull << 32) + o.part_vecs - 1) / o.part_vecs);
    at += bytes;
    return 0;
  };
  for (int64_t k = 0; k < in.num_parts; ++k) {
    const distca_token_part &p = in.part[k];
    if (!p.data) return fail(DISTCA_E_INVALID, "%s: null pointer", what);
    if (!aligned16(p.data) || !aligned16(buffer)) return fail(DISTCA_E_INVALID, "%s: tensor/buffer must be 16-byte aligned", what);
    if (p.bytes <= 0 || p.bytes % 16 || p.pitch < p.bytes || p.pitch % 16 || p.pitch >= (1ll << 31) || at + p.bytes > token_bytes)
      return fail(DISTCA_E_INVALID, "%s: a part of %lld B at a pitch of %lld B in a token of %lld B (multiples of 16)", what, (long long)p.bytes, (long long)p.pitch, (long long)token_bytes);
    if (const int rc = append(p.data, p.pitch, p.bytes)) return rc;
  }
  if (at < token_bytes && to_buffer)
    if (const int rc = append(nullptr, 0, token_bytes - at)) return rc;
  return 0;
}

// The lines between slices and vectors.  Slices have many vectors of a thread in flight and gain on bandwidth, the sooner the less there is to
// be found out on the way: an unpack by vectors cannot ask for anything before the list is read, while a pack has its rows by then; adding rows up, a
// vector has a load in flight at a time.  What slices lose is a trip there and back for each run they walk, so that every line lies further up
// the more shards there are to the slice of a job; rows of several replicas and parts of a few bytes a token (lse of 8 heads) cost slices more than the
// bandwidth gives up to 128 MB.  Of 1134 launches of 16 to 127 MB (4 to 64 heads, 3 to 250 documents) the one chosen is at most 10 % slower than the
// other, 19 times more than 5 %, where one line of 128 MB, 32 MB with sums, took up to 93 % longer.  us by slices / by vectors around the lines (12 documents at 32/8 heads, every replica's mask set once in four, where nothing else is said):
//   one tensor unpacked          24 MB 14.1 / 13.6   32 MB 16.1 / 16.6   48 MB 20.6 / 22.7   64 MB 25.0 / 28.9
//   q, k, v unpacked             32 MB 17.4 / 16.7   48 MB 21.9 / 23.0   120 documents, 40 MB 26.2 / 24.5, 72 MB 35.6 / 39.3
//   one tensor packed            32 MB 16.1 / 15.4   48 MB 20.7 / 20.7   64 MB 25.2 / 26.1
//   [out | lse] unpacked         64 MB 30.3 / 29.3   96 MB 39.6 / 42.2   3 documents, 40 MB 18.7 / 19.5   8/2 heads, 100 documents, 128 MB 69.9 / 59.4
//   gradients, replicas added    48 MB 31.5 / 27.7   64 MB 37.2 / 35.6   72 MB 36.9 / 36.9   96 MB 48.7 / 50.6
//   gradients, copies added      48 MB 26.2 / 24.7   64 MB 30.0 / 31.5   96 MB 39.8 / 43.5
//   q, k, v packed to replicas   64 MB 34.6 / 32.6  128 MB 64.7 / 60.0; the request 64 MB 38.0 / 29.9, 128 MB 61.5 / 54.5
// (One tensor packed, 88 to 127 MB: slices begin a second round of workgroups at 84 MB, and until they fill it vectors gain again, 36.0 / 34.1, 48.6 / 47.1, but
// not where a wave looks through several reads of shards, 250 of them 38.9 / 44.6.)
constexpr int64_t kVectorUnpackBytes = 30 * 1000 * 1000, kVectorPackBytes = 40 * 1000 * 1000, kVectorSumBytes = 50 * 1000 * 1000, kVectorMostBytes = 128ll << 20;
constexpr int64_t kNarrowPartBytes = 128;
// One vector a thread is possible: a vector's number times the vectors of a part stays below 2^32 (Job::magic).
bool vectors_can(const Jobs &jobs, int64_t total) {
  for (int i = 0; i < jobs.n; ++i) {
    const Job &o = jobs.job[i];
    if (o.num_seq > kVectorSeqs || o.num_tokens * o.part_vecs * o.part_vecs >= (1ll << 32)) return false;
  }
  return total <= kVectorMostBytes;
}
// Which of the two for a launch that may take either (tokens_per_wg: of its slices).
bool vectors_gain(const Jobs &jobs, int64_t total, int to_buffer) {
  bool sums = false, replicas = false, parts = false, narrow = false, one_read = true;
  double walked = 0;   // shards, and their replicas, that a slice walks
  for (int i = 0; i < jobs.n; ++i) {
    const Job &o = jobs.job[i];
    const bool adds_replicas = o.kind == DISTCA_JOB_REPLICA_SUM;
    sums |= adds_replicas || o.kind == DISTCA_JOB_COPY_SUM;
    replicas |= o.kind == DISTCA_JOB_REPLICAS;
    parts |= !o.whole();
    narrow |= !o.whole() && o.part_vecs * 16 < kNarrowPartBytes;
    one_read &= o.num_seq <= 64;
    const double w = (double)o.tokens_per_wg * o.num_seq * (adds_replicas ? o.max_cp : 1) / (double)o.num_tokens;
    walked = w > walked ? w : walked;
  }
  if (!sums && (replicas || narrow || (to_buffer && one_read && total > 2 * num_compute_units() * kRoundBytes))) return true;
  const int64_t line = sums ? kVectorSumBytes : to_buffer ? kVectorPackBytes : kVectorUnpackBytes;
  return total <= line * (1 + (parts && !sums ? 1.25 : 0.5) * walked);
}

int launch_exchange(Jobs &jobs, void *buffer, int to_buffer, void *stream, int timer_id, const char *what) {
  if (jobs.n == 0) return DISTCA_OK;
  int64_t total = 0;
  bool sums = false, parts = false;
  for (int i = 0; i < jobs.n; ++i) {
    const Job &o = jobs.job[i];
    total += o.num_tokens * o.part_vecs * 16;
    sums |= o.kind == DISTCA_JOB_REPLICA_SUM || o.kind == DISTCA_JOB_COPY_SUM;
    parts |= !o.whole();
  }
  bool by_vectors = vectors_can(jobs, total);
  int64_t grid[kMaxJobs];   // slices of each job (below the lowest of the lines nothing asks for them)
  if (!by_vectors || total > kVectorUnpackBytes) {
    const int64_t slice = slice_bytes(total);
    for (int i = 0; i < jobs.n; ++i) {
      Job &o = jobs.job[i];
      const bool sum = o.kind == DISTCA_JOB_REPLICA_SUM || o.kind == DISTCA_JOB_COPY_SUM;
      const int64_t round = (sum ? kUnrollSum : o.whole() ? kUnroll : kUnrollParts) * kVecRound;   // one round of the job's own loop
      int64_t per = slice_tokens(slice < round ? slice : round, o.num_tokens, (int64_t)o.part_vecs * 16, &grid[i]);
      if (!o.whole()) {   // a slice's rows lie within 2^30 bytes on both sides (32-bit offsets), and its vectors within the range of `magic`
        const int64_t widest = o.pitch > o.token_bytes ? o.pitch : o.token_bytes;
        const int64_t most = (1ll << 30) / widest < (1ll << 15) ? (1ll << 30) / widest : (1ll << 15);
        if (per > most) per = most < 1 ? 1 : most, grid[i] = (o.num_tokens + per - 1) / per;
      }
      o.tokens_per_wg = (int32_t)per;
    }
    by_vectors = by_vectors && vectors_gain(jobs, total, to_buffer);
  }
  int64_t wg = 0;
  for (int i = 0; i < jobs.n; ++i) {
    Job &o = jobs.job[i];
    o.first_wg = (int32_t)wg;
    wg += by_vectors ? (o.num_tokens * o.part_vecs + kVectorThreads - 1) / kVectorThreads : grid[i];
    if (wg > 0x7fffffff) return fail(DISTCA_E_INVALID, "%s: grid too large", what);
  }
  hipStream_t s = (hipStream_t)stream;
  uint8_t *buf = (uint8_t *)buffer;
  ScopedTimer timer(timer_id, s);
  const dim3 g((unsigned)wg), b(by_vectors ? kVectorThreads : kPackThreads);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, 0, s, jobs, buf); };
  if (by_vectors) launch(to_buffer ? exchange_vectors_kernel<true> : exchange_vectors_kernel<false>);
  else if (to_buffer) launch(sums ? exchange_kernel<true, true, true> : parts ? exchange_kernel<true, true, false> : exchange_kernel<true, false, false>);
  else launch(sums ? exchange_kernel<false, true, true> : parts ? exchange_kernel<false, true, false> : exchange_kernel<false, false, false>);
  return check_launch(what);
}

distca_exchange_job whole_tokens(int64_t kind, void *tensor, const int64_t *seq_offset, const int64_t *seq_tokens, const int8_t *mask,
                                 int64_t num_seq, int64_t token_bytes, int64_t num_tokens, int64_t max_cp) {
  distca_exchange_job j = {};
  j.kind = kind; j.num_parts = 1; j.max_cp = max_cp; j.num_seq = num_seq; j.num_tokens = num_tokens; j.token_bytes = token_bytes;
  j.seq_offset = seq_offset; j.seq_tokens = seq_tokens; j.mask = mask;
  j.part[0].data = tensor; j.part[0].pitch = j.part[0].bytes = token_bytes;
  return j;
}

}  // namespace
}  // namespace distca

using namespace distca;

extern "C" int distca_exchange(const distca_exchange_job *jobs, int32_t num_jobs, void *buffer, int to_buffer, void *stream) {
  if (num_jobs < 0 || num_jobs > DISTCA_EXCHANGE_MAX_JOBS) return fail(DISTCA_E_INVALID, "exchange: %d jobs (0..%d)", num_jobs, DISTCA_EXCHANGE_MAX_JOBS);
  if (num_jobs > 0 && !jobs) return fail(DISTCA_E_INVALID, "exchange: null job list");
  Jobs list;
  list.n = 0;
  for (int i = 0; i < num_jobs; ++i) {
    if (jobs[i].kind < 0 || jobs[i].kind > DISTCA_JOB_COPY_SUM) return fail(DISTCA_E_INVALID, "exchange: unknown kind of job %lld", (long long)jobs[i].kind);
    if (jobs[i].num_parts < 1 || jobs[i].num_parts > DISTCA_TOKEN_MAX_PARTS) return fail(DISTCA_E_INVALID, "exchange: %lld parts (1..%d)", (long long)jobs[i].num_parts, DISTCA_TOKEN_MAX_PARTS);
    const int rc = add_job(&list, jobs[i], jobs[i].token_bytes, to_buffer, buffer, "exchange");
    if (rc) return rc;
  }
  return launch_exchange(list, buffer, to_buffer, stream, DISTCA_TIMER_MEMCPY_NON_CP, "exchange");
}

extern "C" int distca_memcpy_non_cp(void *tensor, void *buffer, const int64_t *seq_offset, const int64_t *seq_tokens,
                                    const int8_t *copy_seq_mask, int64_t num_seq, int64_t token_bytes, int64_t num_tokens,
                                    int to_buffer, void *stream) {
  Jobs list;
  list.n = 0;
  const int rc = add_job(&list, whole_tokens(DISTCA_JOB_PLAIN, tensor, seq_offset, seq_tokens, copy_seq_mask, num_seq, token_bytes, num_tokens, 1),
                         token_bytes, to_buffer, buffer, "memcpy_non_cp");
  return rc ? rc : launch_exchange(list, buffer, to_buffer, stream, DISTCA_TIMER_MEMCPY_NON_CP, "memcpy_non_cp");
}

extern "C" int distca_memcpy_non_cp_multi(const distca_pack_job *jobs, int32_t num_jobs, void *buffer, int to_buffer, void *stream) {
  static_assert(DISTCA_PACK_MAX_JOBS <= DISTCA_EXCHANGE_MAX_JOBS, "one launch");
  if (num_jobs < 0 || num_jobs > DISTCA_PACK_MAX_JOBS) return fail(DISTCA_E_INVALID, "memcpy_non_cp_multi: %d jobs (0..%d)", num_jobs, DISTCA_PACK_MAX_JOBS);
  if (num_jobs == 0) return DISTCA_OK;
  if (!jobs) return fail(DISTCA_E_INVALID, "memcpy_non_cp_multi: null job list");
  Jobs list;
  list.n = 0;
  for (int i = 0; i < num_jobs; ++i) {
    const distca_pack_job &in = jobs[i];
    const int rc = add_job(&list, whole_tokens(DISTCA_JOB_PLAIN, in.tensor, in.seq_offset, in.seq_tokens, in.copy_seq_mask, in.num_seq, in.token_bytes, in.num_tokens, 1),
                           in.token_bytes, to_buffer, buffer, "memcpy_non_cp_multi");
    if (rc) return rc;
  }
  return launch_exchange(list, buffer, to_buffer, stream, DISTCA_TIMER_MEMCPY_NON_CP, "memcpy_non_cp_multi");
}

extern "C" int distca_memcpy_cp(void *tensor, void *buffer, const int8_t *do_shard, const int64_t *seq_offset,
                                const int64_t *seq_tokens, int64_t token_bytes, int64_t num_tokens, int32_t max_cp,
                                int64_t num_seq, int to_buffer, void *stream) {
  Jobs list;
  list.n = 0;
  const int rc = add_job(&list, whole_tokens(DISTCA_JOB_REPLICAS, tensor, seq_offset, seq_tokens, do_shard, num_seq, token_bytes, num_tokens, max_cp),
                         token_bytes, to_buffer, buffer, "memcpy_cp");
  return rc ? rc : launch_exchange(list, buffer, to_buffer, stream, DISTCA_TIMER_MEMCPY_CP, "memcpy_cp");
}

extern "C" int distca_grad_sum(void *data, int dtype, const int32_t *num_copies, const int64_t *copy_start_id,
                               const int64_t *seq_lens, int64_t num_tokens, int64_t hidden, int64_t num_seq,
                               int64_t max_copies, void *stream) {
  if (num_tokens < 0 || hidden < 0 || num_seq < 0 || max_copies < 0) return fail(DISTCA_E_INVALID, "grad_sum: negative size");
  if (num_tokens == 0 || hidden == 0 || num_seq == 0 || max_copies == 0) return DISTCA_OK;
  if (!data || !num_copies || !copy_start_id || !seq_lens) return fail(DISTCA_E_INVALID, "grad_sum: null pointer");
  if (!aligned16(data)) return fail(DISTCA_E_INVALID, "grad_sum: data must be 16-byte aligned");
  const int64_t esz = dtype == DISTCA_DTYPE_F32 ? 4 : 2;
  if (num_seq >= (1ll << 31)) return fail(DISTCA_E_INVALID, "grad_sum: num_seq must be < 2^31");
  int64_t grid;
  const int64_t per = slice_tokens(slice_bytes(num_tokens * hidden * esz), num_tokens, hidden * esz, &grid);
  if (grid > 0x7fffffff) return fail(DISTCA_E_INVALID, "grad_sum: grid too large");
  hipStream_t s = (hipStream_t)stream;
  ScopedTimer timer(DISTCA_TIMER_GRAD_SUM, s);
  switch (dtype) {
    case DISTCA_DTYPE_F32:
      hipLaunchKernelGGL((grad_sum_kernel<float>), dim3((unsigned)grid), dim3(kPackThreads), 0, s, (float *)data, num_copies,
                         copy_start_id, seq_lens, num_tokens, hidden, num_seq, max_copies, per);
      break;
    case DISTCA_DTYPE_F16:
      hipLaunchKernelGGL((grad_sum_kernel<_Float16>), dim3((unsigned)grid), dim3(kPackThreads), 0, s, (_Float16 *)data, num_copies,
                         copy_start_id, seq_lens, num_tokens, hidden, num_seq, max_copies, per);
      break;
    case DISTCA_DTYPE_BF16:
      hipLaunchKernelGGL((grad_sum_kernel<__bf16>), dim3((unsigned)grid), dim3(kPackThreads), 0, s, (__bf16 *)data, num_copies,
                         copy_start_id, seq_lens, num_tokens, hidden, num_seq, max_copies, per);
      break;
    default:
      return fail(DISTCA_E_UNSUPPORTED, "grad_sum: dtype %d (only fp32, fp16, bf16)", dtype);
  }
  return check_launch("grad_sum");
}
