// Row-wise argmax with clamping, gfx950.
//
// Stands for the token selection at the end of every speculator step,
//   last_tokens = torch.argmax(logits, dim=-1); last_tokens.clamp_(0, vocab_size - 1)
// (arctic_inference/vllm/spec_dec/arctic_speculator.py:846-848, 862), with torch's rules for the winner:
// the largest value, the lowest index among equal values, and a NaN beats every number (the first NaN wins).
//
// A workgroup walks a row, or a segment of one, in 16-byte chunks with streaming loads; every lane keeps its own
// (value, index) winner; winners are merged inside the wave with lane exchanges, across the waves through LDS and,
// where a row is split over several workgroups, across those through a workspace (merge_segments below).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <random>

#include "common.hpp"

namespace arctic {

// A candidate as one 64-bit key whose unsigned order is torch's order of winners (GreaterOrNan with the index as tie
// break, aten/src/ATen/native/SharedReduceOps.h): the value's bits mapped monotonically to an unsigned number in the
// upper half (-0 counts as +0, every NaN as the largest number of all), the complement of the index in the lower half
// (among equal values the lowest index is the largest key).  0 = nothing seen: no element maps to upper half 0.
// Merging two candidates is then one 64-bit unsigned maximum instead of a cascade of floating-point cases.
__device__ __forceinline__ uint64_t winner_key(float value, int index) {
  if (index < 0) return 0;
  uint32_t b = __float_as_uint(value);
  if (b == 0x80000000u) b = 0;   // -0 -> +0 (on the bits: no arithmetic that a denormal mode could touch)
  uint32_t o = b ^ ((b & 0x80000000u) ? 0xffffffffu : 0x80000000u);
  if (value != value) o = 0xffffffffu;
  return ((uint64_t)o << 32) | (uint32_t)~(uint32_t)index;
}
__device__ __forceinline__ int winner_index(uint64_t key) { return key ? (int)~(uint32_t)key : -1; }

// The wave's winner in every lane, in two 32-bit passes: the largest upper half, then the largest lower half among the
// candidates that have it.  A step of a pass is one v_max_u32 with a DPP operand (the 64-bit maximum it stands for
// takes two moves, a compare and two selects): partners at distance 1 and 2 inside a quad, then the mirrored half and
// the mirrored row of 16 lanes, then the row in front and the two rows in front broadcast into the next ones, which
// leaves the wave's maximum in lane 63.  kRows = 1: only lanes 0 ... 15 hold candidates.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t max_dpp(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRowMask, 0xf, kRowMask == 0xf));
}
template <int kRows>
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = max_dpp<0xB1, 0xf>(v);    // quad_perm [1,0,3,2]
  v = max_dpp<0x4E, 0xf>(v);    // quad_perm [2,3,0,1]
  v = max_dpp<0x141, 0xf>(v);   // row_half_mirror
  v = max_dpp<0x140, 0xf>(v);   // row_mirror
  if constexpr (kRows == 1) return (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
  v = max_dpp<0x142, 0xa>(v);   // row_bcast15 into rows 1 and 3
  v = max_dpp<0x143, 0xc>(v);   // row_bcast31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
template <int kRows = 4>
__device__ __forceinline__ uint64_t wave_winner(uint64_t k) {
  const uint32_t value = (uint32_t)(k >> 32);
  const uint32_t top = wave_max<kRows>(value);
  const uint32_t index = wave_max<kRows>(value == top ? (uint32_t)k : 0u);
  return ((uint64_t)top << 32) | index;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

struct F32Elem {
  static constexpr int kPerChunk = 4;
  // NaN exactly when the chunk holds a NaN or infinities of both signs
  __device__ static __forceinline__ float probe(const uint4 &v) {
    return (__uint_as_float(v.x) + __uint_as_float(v.y)) + (__uint_as_float(v.z) + __uint_as_float(v.w));
  }
  __device__ static __forceinline__ void unpack(const uint4 &v, float (&f)[8]) {
    f[0] = __uint_as_float(v.x);
    f[1] = __uint_as_float(v.y);
    f[2] = __uint_as_float(v.z);
    f[3] = __uint_as_float(v.w);
  }
  __device__ static __forceinline__ float one(const void *p, int64_t i) { return ((const float *)p)[i]; }
};
template <typename T>
struct HalfElem {
  static constexpr int kPerChunk = 8;
  // the sum of the chunk's eight values, two per instruction straight from the packed words (v_dot2c_f32_bf16 /
  // v_dot2c_f32_f16 with a vector of ones): NaN exactly when the chunk holds a NaN or infinities of both signs
  __device__ static __forceinline__ float probe(const uint4 &v) {
    float acc = 0.f;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (T::kCode == ARCTIC_DTYPE_BF16) {
        const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};
        acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w[k]), ones, acc, false);
      } else {
        const f16x2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, w[k]), ones, acc, false);
      }
    }
    return acc;
  }
  __device__ static __forceinline__ void unpack(const uint4 &v, float (&f)[8]) { unpack8<T>(v, f); }
  __device__ static __forceinline__ float one(const void *p, int64_t i) {
    return T::lo((uint32_t)((const uint16_t *)p)[i]);
  }
};

// kVec: the body of a row, from its first 16-byte boundary on, is read in 16-byte chunks; the elements in front of
// that boundary (a row pitch that is no multiple of 16 bytes puts every row somewhere else), those behind the last
// whole chunk, and everything when !kVec (a pointer that is not even element-aligned) are read one by one.
// kUnroll chunks per lane form a batch;
// kLockstep: a workgroup barrier (no memory wait) behind every batch's requests, so that every wave of the row has
// asked for batch k before any wave asks for batch k + 1 (a CU serves its oldest wave first: without the barrier the
// oldest wave runs through all its batches before the youngest gets its first one in).
// kHead: rows may start between two 16-byte boundaries (without it the host has checked that none does).
// Returns the winner of the `cols` elements at `row` as a key whose index counts from `first`, in every lane of wave 0 of
// a workgroup of `lanes`.
template <typename Elem, bool kVec, int kUnroll, bool kLockstep, bool kHead>
__device__ __forceinline__ uint64_t find_winner(const char *__restrict__ row, int cols, int first, int lanes) {
  __shared__ uint64_t wave_key[16];
  // Per lane: the largest number seen, the chunk it was first seen in and that chunk's words (a strict ">" keeps the
  // earlier of equal values, the lane's chunk indices only grow); which of the chunk's elements it was is worked out
  // once, after the loop.  Apart from that the first NaN: a chunk's sum is NaN only if the chunk holds a NaN (or
  // infinities of both signs), so the per-element NaN test runs almost never.
  constexpr int P = Elem::kPerChunk;
  const int head = kVec && kHead ? min(cols, (int)((0 - (uintptr_t)row) & 15) / (16 / P)) : 0;   // elements in front of the body
  const int chunks = kVec ? (cols - head) / P : 0;
  const char *body = row + (int64_t)head * (16 / P);
  float best = -__builtin_inff();
  int best_at = -1;
  int nan_at = 0x7fffffff;
  auto number = [&](float v, int i) {
    if (v > best) {
      best = v;
      best_at = i;
    }
  };
  // a lane's candidates come in the order of their indices (head, chunks, tail), so that ">" keeps the first of equals
  if ((int)threadIdx.x < head) {
    const float v = Elem::one(row, threadIdx.x);
    best_at = threadIdx.x;   // stands for the lane even when it is -inf: a row of -inf must answer 0
    best = v == v ? v : best;
    if (v != v) nan_at = threadIdx.x;
  }
  int done = 0;
  if (kVec) {
    int best_chunk = -1;
    uint4 best_words = make_uint4(0, 0, 0, 0);
    const int stride = kUnroll * lanes;
    auto request = [&](int c0, uint4 (&raw)[kUnroll]) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int c = c0 + u * lanes;
        if (c < chunks) raw[u] = load16_stream(body + (int64_t)c * 16);
      }
    };
    auto look_at_chunk = [&](int c, const uint4 &words) {
      float f[8];
      Elem::unpack(words, f);
      float top = best;   // fmaxf drops NaNs: they are found through the sum below
#pragma unroll
      for (int j = 0; j < P; j += 2) top = fmaxf(fmaxf(top, f[j]), f[j + 1]);
      if (top > best) {
        best_chunk = c;
        best_words = words;
      }
      best = top;
      const float sum = Elem::probe(words);
      if (sum != sum) {
#pragma unroll
        for (int j = 0; j < P; ++j)
          if (f[j] != f[j]) nan_at = min(nan_at, head + c * P + j);
      }
    };
    auto look_at = [&](int c0, const uint4 (&raw)[kUnroll]) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int c = c0 + u * lanes;
        if (c < chunks) look_at_chunk(c, raw[u]);
      }
    };
    if constexpr (kLockstep) {
      const int batches = (chunks + stride - 1) / stride;   // the same for every wave, as the barrier needs it
      int c0 = threadIdx.x;
      for (int b = 0; b < batches; ++b, c0 += stride) {
        uint4 raw[kUnroll];
        request(c0, raw);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        look_at(c0, raw);
      }
    } else {
      int c0 = threadIdx.x;
      for (; c0 < chunks; c0 += stride) {
        uint4 raw[kUnroll];
        request(c0, raw);
        look_at(c0, raw);
      }
    }
    done = head + chunks * P;
    if (best_chunk >= 0) {
      // the first element of that chunk that equals the lane's maximum
      float f[8];
      Elem::unpack(best_words, f);
      int j = P - 1;
#pragma unroll
      for (int k = P - 2; k >= 0; --k)
        if (f[k] == best) j = k;
      best_at = head + best_chunk * P + j;
    } else if (best_at < 0 && (int)threadIdx.x < chunks) {
      best_at = head + (int)threadIdx.x * P;   // nothing above -inf here: the lane's first element stands for its chunks
    }
  }
  // (a lane without chunks takes its first tail element, if it has one, the same way: a row of -inf must answer 0)
  if (best_at < 0 && done + (int)threadIdx.x < cols) best_at = done + (int)threadIdx.x;
  for (int i = done + threadIdx.x; i < cols; i += lanes) {
    const float v = Elem::one(row, i);
    number(v, i);
    if (v != v) nan_at = min(nan_at, i);
  }
  uint64_t w = nan_at != 0x7fffffff ? winner_key(__builtin_nanf(""), first + nan_at)
                                    : winner_key(best, best_at < 0 ? -1 : first + best_at);

  w = wave_winner(w);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) wave_key[wave] = w;
  __syncthreads();
  if (wave > 0) return 0;
  const int waves = lanes >> 6;
  return wave_winner<1>(lane < waves ? wave_key[lane] : 0);   // at most 16 waves
}

__device__ __forceinline__ void store_winner(int64_t *out, uint64_t key, int64_t max_index) {
  const int found = winner_index(key);
  const int64_t idx = found < 0 ? 0 : found;
  *out = idx > max_index ? max_index : idx;
}

struct Segment {
  uint64_t key;
  uint64_t seal;
};
static_assert(sizeof(Segment) == ARCTIC_ARGMAX_SEGMENT_BYTES, "the workspace holds one Segment per workgroup");

struct ArgmaxParams {
  int64_t *out;
  const char *in;
  int64_t row_stride_bytes;
  int64_t max_index;
  int cols;
  int lanes;   // of a workgroup
  // rows split over several workgroups:
  int segment, parts;
  uint64_t call;
  Segment *workspace;
};

template <typename Elem, bool kVec, int kUnroll = 4, bool kLockstep = false, bool kHead = false>
__global__ __launch_bounds__(1024) void row_argmax_kernel(const ArgmaxParams p) {
  const uint64_t w = find_winner<Elem, kVec, kUnroll, kLockstep, kHead>(p.in + (int64_t)blockIdx.x * p.row_stride_bytes,
                                                                        p.cols, 0, p.lanes);
  if (threadIdx.x == 0) store_winner(p.out + blockIdx.x, w, p.max_index);
}

// ---- rows split over several workgroups ----------------------------------------------------------------------
// One workgroup pulls at most about 50 GB/s out of HBM (what a CU keeps outstanding over the latency), 5 us for the
// 256 KB of a row of 128256 16-bit logits, so a few rows leave the chip idle.  Here each row is cut into `parts`
// segments of at least two chunks per lane.  Every workgroup leaves its segment's winner in the workspace and then reads
// the winners of the whole row; a workgroup that finds all of them there merges them and stores the row's answer.
//
// The workspace is memory of the call's own with unknown contents: nothing has to be cleared beforehand and nothing is
// shared between calls.  A winner counts as there when the word beside it is its seal, a bijection of the winner and of
// a number that no other call has (64 bits from a generator seeded by the system), so what the memory held before
// passes for a winner with a probability of 2^-64, and a half-written pair does not pass at all.  The workgroups that
// answer break the row's seals, so that a graph that is replayed, with the same number, starts without any.
//
// Some workgroup always finds the row complete: every one waits until its own pair has been stored before it reads,
// so the one whose pair is stored last sees all of them, unless another has answered already and broken the seals.
// Several may answer; they store the same value.  No workgroup waits for another.  Stores and loads of the workspace
// are agent-scope atomics, which go to the memory all XCDs see whatever their L2s hold, so the wait for the stores'
// acknowledgement is all the order that is needed; a sequentially consistent fence in its place writes back and
// invalidates the L2 once per workgroup, and those queue up (64 rows of 16 segments: 22.3 us instead of 7.0).
__device__ __forceinline__ uint64_t seal_of(uint64_t key, uint64_t call) { return (key * 0x9E3779B97F4A7C15ull) ^ call; }
__device__ __forceinline__ void share(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t shared(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// By wave 0 of the workgroup, `parts` at most 64.
__device__ __forceinline__ void merge_segments(int64_t *out, Segment *row, int part, int parts, uint64_t key,
                                               uint64_t call, int64_t max_index) {
  const int lane = threadIdx.x;
  if (lane == 0) {
    share(&row[part].key, key);
    share(&row[part].seal, seal_of(key, call));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the pair is stored (comment above)
  uint64_t theirs = 0;
  bool there = true;
  if (lane < parts) {
    theirs = shared(&row[lane].key);
    there = shared(&row[lane].seal) == seal_of(theirs, call);
  }
  if (!__all(there)) return;
  const uint64_t w = wave_winner(theirs);
  if (lane == 0) store_winner(out, w, max_index);
  if (lane < parts) share(&row[lane].seal, ~seal_of(theirs, call));
}

constexpr int kSplitLanes = 512;

template <typename Elem, bool kHead>
__global__ __launch_bounds__(kSplitLanes) void row_argmax_split_kernel(const ArgmaxParams p) {
  const unsigned row = blockIdx.x / (unsigned)p.parts;
  const int part = (int)(blockIdx.x - row * (unsigned)p.parts);
  const int first = part * p.segment;
  const char *at = p.in + (int64_t)row * p.row_stride_bytes + (int64_t)first * (16 / Elem::kPerChunk);
  const uint64_t w = find_winner<Elem, true, 4, false, kHead>(at, min(p.segment, p.cols - first), first, kSplitLanes);
  if (threadIdx.x < 64)
    merge_segments(p.out + row, p.workspace + (int64_t)row * p.parts, part, p.parts, w, p.call, p.max_index);
}

}  // namespace arctic

using namespace arctic;

// How many workgroups share a row (1: not split), and the elements of each one's segment.  The exchange costs about
// a microsecond (store, acknowledgement, read), so a row is split where that buys more (calls in graphs, both sides in turn,
// their inputs one after the other out of 800 MB and more, of the smallest 96 sets):
//  - up to 128 rows, which leave CUs idle: the more rows the longer they have to be, from 85 on 180 chunks of 16 bytes for each
//    row but 5100.  Eight segments against one, in per cent, aligned rows / others: bf16 74 rows of 10240 chunks -9 / -4, 80 of
//    11000 -5 / -4, 85 of 12000 -4 / -4, 96 of 12000 -3 / -1, of 11000 -2 / -1, 100 of 13500 -10 / -5, of 12000 +1 / +3, 112 of
//    15500 -7 / -5, of 12500 -1 / +3, 128 of 17500 -4 / -2, of 18992 +1 / -3, of 12500 +2 / +4; fp32 74 of 10240 -5 / -2, 85 of
//    12000 -1 / -3, 96 of 12500 -6 / -4, of 11000 +2 / 0, 112 of 15500 -5 / -4, of 18992 +2 / -5, 128 of 19500 -2 / -2, of 14000
//    +3 / 0.  Up to 48 rows of 16-bit logits from 8192 chunks on (20 of 8192 -15 / -15, 41 -7 / +2, 48 -6 / +2, 64 -2 / +3); fp32
//    rows, whose chunks are half as much work, from 10240 (1 of 8192 3.74 us / 4.22 where the L2 holds the inputs, from HBM 4.34
//    / 3.88);
//  - a few more rows than one or two for every CU, where some CUs would do twice or half as much again as the others: up to 304
//    from 12288 chunks on (bf16, per cent against one workgroup per row: 257 rows of 12288 -6, of 18992 -2, of 24576 -9, of 10000
//    -1, 288 of 12288 -4, 304 of 12288 -2, of 18992 0, of 24576 -4, 320 of 12288 0, of 18992 +2), fp32 beyond 288 rows from 24576
//    (257 of 12288 -1, 288 0, 296 +1, 304 +2, of 18992 +2, of 24576 -2, of 32768 -3); up to 600 from 10000 (bf16 513 of 10000 -6, 600
//    of 10000 0, of 10500 -5, of 16032 -2, 616 of 10000 +1; fp32 513 of 10000 -3, 600 of 10000 -1, of 16032 0); up to 704 from 28672,
//    of which the upper half is level (bf16 640 of 28672 -2, of 32768 -6, 704 of 28672 +2, of 32768 -2, of 40960 +2, of 65536 -2; fp32
//    640 of 30720 -2, 704 of 28672 +1, of 32768 -1, of 40960 +4, of 65536 -3).
//    Only where every row starts on a 16-byte boundary: others lose up to a quarter below 14000 chunks (257 x 80001 +18, 272 x
//    98305 +9, 513 x 80001 +19) and are level about 16032 (257 rows +4, 272 0, 304 +3, 513 0, 600 +1).
// Up to sixteen segments of 1024 chunks or more while they make no more than two workgroups per CU (7 x 128256: 32 segments 4.7
// us, 16 4.4), and not fewer than eight, of very long rows six (85 x 128256 six 7.93, eight 7.47, sixteen 8.08; 78 x 262144 six
// 10.3, eight 10.8).  Workgroups of 256 and 1024 lanes are 0.1-0.2 us slower.
static int argmax_parts(bool aligned_rows, int64_t rows, int cols, int dtype, int *segment) {
  constexpr int64_t kMostParts = 16, kParts = 8, kWorkgroups = 512, kMinChunksPerPart = 1024;
  *segment = cols;
  const int64_t chunks = dtype == ARCTIC_DTYPE_F32 ? cols / 4 : cols / 8;
  int64_t parts = 1;
  const int64_t shortest = dtype == ARCTIC_DTYPE_F32 ? 10240 : rows <= 48 ? 8192 : 10000;
  if (rows > 0 && rows <= 128 && chunks >= std::max(shortest, 180 * rows - 5100)) {
    parts = std::min({kMostParts, chunks / kMinChunksPerPart, kWorkgroups / rows});
    if (parts < (chunks < 18000 ? kParts : 6)) parts = kParts;
  } else if (aligned_rows &&
             ((rows > 256 && rows <= 304 && chunks >= (dtype == ARCTIC_DTYPE_F32 && rows > 288 ? 24576 : 12288)) ||
              (rows > 512 && rows <= (chunks >= 28672 ? 704 : 600) && chunks >= 10000))) {
    parts = kParts;
  }
  if (parts == 1) return 1;
  *segment = (int)((cols + parts - 1) / parts + 63) & ~63;   // whole 128-byte lines of an aligned row
  return (cols + *segment - 1) / *segment;
}

static bool rows_on_16_bytes(const void *logits, int64_t rows, int64_t row_stride, int dtype) {
  const uint64_t pitch = (uint64_t)row_stride * (dtype == ARCTIC_DTYPE_F32 ? 4 : 2);
  return (uintptr_t)logits % 16 == 0 && (pitch % 16 == 0 || rows == 1);
}

static int64_t argmax_workspace(bool aligned_rows, int64_t rows, int cols, int dtype) {
  int segment;
  const int parts = argmax_parts(aligned_rows, rows, cols, dtype, &segment);
  return parts > 1 ? rows * parts * (int64_t)sizeof(Segment) : 0;
}
extern "C" int64_t arctic_argmax_workspace_bytes(int64_t rows, int cols, int dtype) {
  return argmax_workspace(true, rows, cols, dtype);   // what is split wherever its rows start is split the same aligned
}
extern "C" int64_t arctic_argmax_workspace_bytes_at(const void *logits, int64_t rows, int cols, int64_t row_stride, int dtype) {
  if ((uintptr_t)logits % (dtype == ARCTIC_DTYPE_F32 ? 4 : 2)) return 0;   // element by element, one workgroup per row
  return argmax_workspace(rows_on_16_bytes(logits, rows, row_stride, dtype), rows, cols, dtype);
}

// A number per call that no other call has: a 64-bit counter from a seed the system draws, spread by an odd factor.
static uint64_t call_number() {
  static std::atomic<uint64_t> next{((uint64_t)std::random_device{}() << 32) ^ std::random_device{}()};
  return next.fetch_add(1, std::memory_order_relaxed) * 0xD1342543DE82EF95ull;
}

extern "C" int arctic_argmax_clamp(int64_t *out, const void *logits, int64_t rows, int cols, int64_t row_stride,
                                   int64_t max_index, int dtype, void *stream) {
  return arctic_argmax_clamp_split(out, logits, rows, cols, row_stride, max_index, dtype, nullptr, 0, stream);
}

extern "C" int arctic_argmax_clamp_split(int64_t *out, const void *logits, int64_t rows, int cols, int64_t row_stride,
                                         int64_t max_index, int dtype, void *workspace, int64_t workspace_bytes,
                                         void *stream) {
  const char *fn = "argmax_clamp";
  if (dtype != ARCTIC_DTYPE_F32 && dtype != ARCTIC_DTYPE_F16 && dtype != ARCTIC_DTYPE_BF16)
    return fail(ARCTIC_ERR_UNSUPPORTED, "%s: logits must be fp32, fp16 or bf16", fn);
  if (rows < 0 || rows > 0x7fffffffLL || cols <= 0 || max_index < 0 || row_stride < 0)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: rows >= 0, cols > 0, max_index >= 0 and a non-negative pitch are required",
                fn);
  if (rows == 0) return ARCTIC_OK;
  if (!out || !logits) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null tensor pointer", fn);
  const int es = dtype == ARCTIC_DTYPE_F32 ? 4 : 2;
  if (cols > (1 << 30) || !pitch_ok(row_stride, rows, es))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: more than 2^30 columns, or a row pitch out of range", fn);
  const int64_t stride_bytes = row_stride * es;
  const bool vec = (uintptr_t)logits % es == 0;   // rows may start anywhere between two 16-byte boundaries
  const bool aligned_rows = rows_on_16_bytes(logits, rows, row_stride, dtype);
  const int per_chunk = 16 / es;
  hipStream_t s = (hipStream_t)stream;
  int segment;
  const int parts = argmax_parts(aligned_rows, rows, cols, dtype, &segment);
  if (vec && parts > 1 && workspace) {
    if ((uintptr_t)workspace % 8 || workspace_bytes < rows * parts * (int64_t)sizeof(Segment))
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: the workspace must be 8-byte aligned and hold %lld bytes", fn,
                  (long long)(rows * parts * (int64_t)sizeof(Segment)));
    const ArgmaxParams p = {out, (const char *)logits, stride_bytes, max_index, cols, kSplitLanes, segment, parts,
                            call_number(), (Segment *)workspace};
#define ARCTIC_ARGMAX_SPLIT(ELEM, HEAD) \
  launch(row_argmax_split_kernel<ELEM, HEAD>, dim3((unsigned)(rows * parts)), kSplitLanes, s, p)
    if (dtype == ARCTIC_DTYPE_F32) {
      if (aligned_rows) ARCTIC_ARGMAX_SPLIT(F32Elem, false);
      else ARCTIC_ARGMAX_SPLIT(F32Elem, true);
    } else if (dtype == ARCTIC_DTYPE_BF16) {
      if (aligned_rows) ARCTIC_ARGMAX_SPLIT(HalfElem<BF16>, false);
      else ARCTIC_ARGMAX_SPLIT(HalfElem<BF16>, true);
    } else {
      if (aligned_rows) ARCTIC_ARGMAX_SPLIT(HalfElem<F16>, false);
      else ARCTIC_ARGMAX_SPLIT(HalfElem<F16>, true);
    }
#undef ARCTIC_ARGMAX_SPLIT
    return check_launch(fn);
  }
  int threads = (int)std::min<int64_t>(1024, std::max<int64_t>(64, ((cols / per_chunk / 4 + 63) / 64) * 64));
  const dim3 grid((unsigned)rows);
  // Two workgroups on a CU (its 2048 lanes hold no third) keep their waves in step, a chunk at a time: they then finish
  // together with little left to do.  A row of one batch (four chunks for each of 1024 lanes) only loses by asking for one chunk
  // at a time, and beyond 512 rows a workgroup that ends early lets the next one begin, which steps prevent.  In step against
  // not, per cent per call in a graph (inputs as above), lowest and highest of bf16 and fp32 rows, aligned and not: 257 to 512 rows
  // of 2000 chunks of 16 bytes +7 and +22, of 3000 0 and +12, of 3600 to 4096 of bf16 and of more than 384 rows -4 and +4, of 270 to
  // 350 fp32 rows of 3600 to 4096 -6 and +1 (mean -3), of 4097 -5 and +4, of 5000 -11 and -3, of 9000 -12 and -2, of 16032 -12 and 0, of
  // 32768 -18 and -6; 513 to 704 rows of up to 28672 chunks +3 and +22; 768 rows +1 and +14, of 32768 chunks alone -5 and -2 (of
  // 30720 and 36000 0 and +4).  Where nearly every CU has two workgroups and rows are not quite two batches long it hangs on each
  // length: of 2400 drawn launches of 421 to 512 rows the mean of aligned rows / others is +0.8 / +0.8 at 4097 to 4300 chunks, -0.4 /
  // -0.9 to 4700, -3.8 / -2.3 to 6100, -1.9 / -0.6 to 6300, -1.5 / -0.2 to 7100, -0.4 / +0.9 to 7700, -1.2 / +0.2 to 8300, -0.6 / +1.0 to 8700,
  // -2.8 / -1.9 to 9500, so that only others of 6200 to 8192, which include 50257 columns (+1.8), go without.
  const int chunks = cols / per_chunk;
  const bool not_quite_two = !aligned_rows && rows > 420 && chunks >= 6200 && chunks <= 8192;
  const int shortest = dtype == ARCTIC_DTYPE_F32 && rows <= 384 ? 3600 : 4097;
  const bool lockstep = rows > 256 && rows <= 512 && chunks >= shortest && !not_quite_two;
  const ArgmaxParams p = {out, (const char *)logits, stride_bytes, max_index, cols, threads, cols, 1, 0, nullptr};
#define ARCTIC_ARGMAX_KERNEL(...) launch(row_argmax_kernel<__VA_ARGS__>, grid, threads, s, p)
#define ARCTIC_ARGMAX_LAUNCH(ELEM)                                                       \
  do {                                                                                   \
    if (!vec) ARCTIC_ARGMAX_KERNEL(ELEM, false);                                         \
    else if (!aligned_rows && lockstep) ARCTIC_ARGMAX_KERNEL(ELEM, true, 1, true, true); \
    else if (!aligned_rows) ARCTIC_ARGMAX_KERNEL(ELEM, true, 4, false, true);            \
    else if (lockstep) ARCTIC_ARGMAX_KERNEL(ELEM, true, 1, true);                        \
    else ARCTIC_ARGMAX_KERNEL(ELEM, true);                                               \
  } while (0)
  if (dtype == ARCTIC_DTYPE_F32) ARCTIC_ARGMAX_LAUNCH(F32Elem);
  else if (dtype == ARCTIC_DTYPE_BF16) ARCTIC_ARGMAX_LAUNCH(HalfElem<BF16>);
  else ARCTIC_ARGMAX_LAUNCH(HalfElem<F16>);
#undef ARCTIC_ARGMAX_LAUNCH
#undef ARCTIC_ARGMAX_KERNEL
  return check_launch(fn);
}
