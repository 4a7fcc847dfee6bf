// Fused LSTM-style gate / cell / state update of the Arctic speculator, gfx950.
//
// Replaces sum_lstm_cuda and its kernels
// (csrc/custom_ops/sum_lstm.cu:14-473 in the reference).
//
// One workgroup per row (few long rows: several, which share its last phase).  On the vector paths each lane owns 16-byte chunks
// (8 elements) at the same column of all four gates of `states` and `z4` and of
// `prev_cell`: nine 16-byte loads per chunk.  The row then stays in registers
// across both RMS reductions, so HBM sees 9*D elements read and 2*D written per
// row (the reference re-reads the cell gate and reads out_cell back: 12*D).
// Sums are DPP wave reductions plus an LDS combine.  Three kernels:
// sum_lstm_staged_kernel (rows of up to 8192 elements: the nine loads are
// requested in stages, between the stages of the arithmetic, or, for few short rows, ahead of it; one chunk per lane),
// sum_lstm_vec_kernel (the loads requested together: rows of up to 16384 elements
// with two chunks per lane, and short ones without all vectors) and sum_lstm_scalar_kernel (what is left: short rows
// that are not 16-byte aligned and more than 16384 elements, element by element).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "activations.hpp"
#include "common.hpp"

namespace arctic {

// A launch's arguments (common.hpp has what their size costs): 112 bytes with pitches and rows of 32 bits, as the vector
// kernels take them, 120 with an embedding lookup.
template <typename Size>
struct LstmParams {
  char *out_state;
  char *out_cell;
  const char *states;
  const char *z4;
  const char *prev_cell;
  const char *w_cell;
  const char *b_cell;
  const char *w_state;
  const char *b_state;
  Size s_stride;   // all strides in elements
  Size z_stride;
  Size pc_stride;
  Size out_stride;
  Size z_rows;     // rows of z4 when z_index is given; an index is clamped into [0, z_rows)
  int D;
  float inv_D;     // 1 / D
  float alpha;
  float eps_cell;
  float eps_state;
};
template <typename Size>
struct LstmSharedParams : LstmParams<Size> {
  const int64_t *z_index;  // row of z4 to use for each row (an embedding lookup); nullptr = the row itself
};
template <bool kSharedZ>
using LstmParamsOf = std::conditional_t<kSharedZ, LstmSharedParams<uint32_t>, LstmParams<uint32_t>>;
using LstmCall = LstmSharedParams<int64_t>;   // what an entry point was given
template <bool kSharedZ>
struct LstmPartsParams : LstmParamsOf<kSharedZ> {
  int rows;   // the grid's first dimension is rounded up
};
template <bool kSharedZ, bool kParts>
using LstmStagedParams = std::conditional_t<kParts, LstmPartsParams<kSharedZ>, LstmParamsOf<kSharedZ>>;

// The row of z4 that a row adds.
template <bool kSharedZ, typename Params>
__device__ __forceinline__ int64_t z_row_of(const Params &p, int64_t row) {
  if constexpr (kSharedZ)
    if (p.z_index) return min(max(p.z_index[row], (int64_t)0), (int64_t)p.z_rows - 1);
  return row;
}

// The index of that row as it was given, by a load that nothing waits for yet (without indices of the arguments themselves).
template <typename Params>
__device__ __forceinline__ int64_t z_id_of(const Params &p, int64_t row) {
  typedef const __attribute__((address_space(4))) int64_t *Constant;
  const uintptr_t none = (uintptr_t)(const void *)__builtin_amdgcn_kernarg_segment_ptr();
  return *(Constant)(p.z_index ? (uintptr_t)(p.z_index + row) : none);
}

// kFullWaves: rows 16-byte aligned, all four scale / shift vectors given, every lane of every wave owns a chunk of 8
// elements; kRagged: the same with lanes to spare in the last wave; kAnyRow: everything else - vectors missing, rows
// only element-aligned (odd widths, pitches or bases; see common.hpp).
enum RowKind { kFullWaves, kRagged, kAnyRow };

// kSharedZ: `z4` holds ONE gate-wide row per token ([rows, D]) that is added to all four
// gates, as the speculator's z4 = emb.repeat(1, 1, 4) would; it is then read once, not four times.
// A null prev_cell stands for a cell of zeros.  Absent scale / shift vectors stand for 1 / 0, which is exact: the norm
// is one multiply and one fused multiply-add per element whichever vectors were given.  Every lane then reads the same
// chunk of ones or zeros below, which leaves the kernels without a branch between a row's requests (one there costs
// 0.25 us at 512 rows of 4096: requests in front of it are waited for behind it).  kMayMiss: a vector can be absent.
__constant__ const uint32_t kChunkOfZeros[4] = {0, 0, 0, 0};
__constant__ const uint32_t kChunkOfOnesF16[4] = {0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
__constant__ const uint32_t kChunkOfOnesBF16[4] = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
template <typename T, bool kMayMiss>
__device__ __forceinline__ Chunk load_scale(const char *w, uint32_t off) {
  if constexpr (!kMayMiss) return Chunk::load(w + off);
  const char *ones = (const char *)(T::kCode == ARCTIC_DTYPE_BF16 ? kChunkOfOnesBF16 : kChunkOfOnesF16);
  return Chunk::load<true>((w ? w : ones) + (w ? off : 0u));
}
template <bool kMayMiss>
__device__ __forceinline__ Chunk load_shift(const char *b, uint32_t off) {
  if constexpr (!kMayMiss) return Chunk::load(b + off);
  return Chunk::load<true>((b ? b : (const char *)kChunkOfZeros) + (b ? off : 0u));
}

// Rows beyond one chunk per lane of 1024 lanes, with two of them, and rows of up to 2048 elements that lack a
// scale or shift vector, with one (launch_lstm has the rule).  Loads are issued in the order in which the arithmetic needs them -
// cell gate, forget gate, previous cell, input gate, output gate - and memory returns them in that order, so the first
// row sum, the candidate GELU and the early sigmoids run while the later gates are still on their way, and only one
// sigmoid, one multiply and the store remain after the last load has landed.
// kBare: none of the four vectors is given, and nothing stands in for them (us per call in a graph, ones and zeros read /
// not read: 64 rows of 12288 with one z for all gates 10.9 / 9.9, 300 of 16384 29.0 / 26.4).
template <int K>
struct LstmRow {
  Chunk sc[K], zc[K], sf[K], zf[K], si[K], zi[K], pc[K], so[K], zo[K];
};

template <typename T, int K, bool kFastGelu, bool kSharedZ, bool kAnyAlignment, bool kBare>
__global__ __launch_bounds__(K == 1 ? 256 : 1024) void sum_lstm_vec_kernel(const LstmParamsOf<kSharedZ> p) {
  __shared__ float slots_cpre[16];
  __shared__ float slots_cnew[16];
  constexpr int E = Chunk::kElems;
  using C = Chunk;
  const int D = p.D;
  const int64_t gate_bytes = (int64_t)D * 2;
  Place at[K];
  const int waves = (((D + 7) / 8 + K - 1) / K + 63) / 64;   // of the workgroup, as launched
#pragma unroll
  for (int k = 0; k < K; ++k) at[k] = Place(threadIdx.x + k * waves * 64, D);
  auto load = [](const char *q) { return C::load_stream<kAnyAlignment>(q); };
  auto vector = [](const C &given, float (&f)[E], float absent) {
    if constexpr (!kBare) given.template unpack<T>(f);
#pragma unroll
    for (int j = 0; j < E && kBare; ++j) f[j] = absent;
  };

  C wc[K], bc[K], ws[K], bs[K];
  // The scale / shift vectors are the same for every row (cache resident).  They
  // are requested first: memory returns loads in issue order, so asking for them
  // later would park the arithmetic behind the whole row.
#pragma unroll
  for (int k = 0; k < K && !kBare; ++k) {
    wc[k] = load_scale<T, true>(p.w_cell, at[k].off);
    bc[k] = load_shift<true>(p.b_cell, at[k].off);
    ws[k] = load_scale<T, true>(p.w_state, at[k].off);
    bs[k] = load_shift<true>(p.b_state, at[k].off);
  }

  const int64_t row = blockIdx.x;
  LstmRow<K> r;
  {
    const char *s_row = p.states + row * p.s_stride * 2;
    const char *z_row = p.z4 + z_row_of<kSharedZ>(p, row) * p.z_stride * 2;
    const char *pc_row = p.prev_cell ? p.prev_cell + row * p.pc_stride * 2 : s_row;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      r.zc[k] = load(z_row + (kSharedZ ? 0 : 3 * gate_bytes) + at[k].off);
      r.sc[k] = load(s_row + 3 * gate_bytes + at[k].off);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      r.sf[k] = load(s_row + at[k].off);
      r.zf[k] = kSharedZ ? r.zc[k] : load(z_row + at[k].off);
    }
    // (the previous cell and both outputs stream like the gates: a launch boundary writes the outputs back anyway,
    // and streaming stores leave the CU earlier - measured on the staged kernel below)
#pragma unroll
    for (int k = 0; k < K; ++k) r.pc[k] = load(pc_row + at[k].off);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      r.si[k] = load(s_row + gate_bytes + at[k].off);
      r.zi[k] = kSharedZ ? r.zc[k] : load(z_row + gate_bytes + at[k].off);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      r.so[k] = load(s_row + 2 * gate_bytes + at[k].off);
      r.zo[k] = kSharedZ ? r.zc[k] : load(z_row + 2 * gate_bytes + at[k].off);
    }
  }

  char *oc_row = p.out_cell + row * p.out_stride * 2;
  char *os_row = p.out_state + row * p.out_stride * 2;
  // phase 1: pre_c and its sum of squares (reference :65-82); needs the cell gate only
  float cact[K][E];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float a[E], b[E];
    r.sc[k].template unpack<T>(a);
    r.zc[k].template unpack<T>(b);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      cact[k][j] = fmaf(p.alpha, b[j], a[j]);
      if (j >= at[k].repeated) ss = fmaf(cact[k][j], cact[k][j], ss);
    }
  }
  const float inv_cpre = rsqrtf(block_sum(ss, slots_cpre, waves) * p.inv_D + p.eps_cell);
  // candidate = gelu(rmsnorm(pre_c)): runs while the other gates are still arriving
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float w[E], b[E];
    vector(wc[k], w, 1.f);
    vector(bc[k], b, 0.f);
#pragma unroll
    for (int j = 0; j < E; ++j) cact[k][j] = gelu<kFastGelu>(fmaf(cact[k][j] * inv_cpre, w[j], b[j]));
  }

  // phase 2: cell update; write out_cell (reference :104-140)
  float cell[K][E];  // ends up as the ROUNDED new cell, as the state phase must see it
  ss = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float a[E], b[E], c[E];
    r.sf[k].template unpack<T>(a);
    r.zf[k].template unpack<T>(b);
    if (!p.prev_cell) r.pc[k] = C::zero();
    r.pc[k].template unpack<T>(c);
#pragma unroll
    for (int j = 0; j < E; ++j) cell[k][j] = sigmoid_f(fmaf(p.alpha, b[j], a[j])) * c[j];
    // keep the forget-gate arithmetic ahead of the wait for the input gate: it then runs while that gate
    // is still arriving instead of in the short stretch between the last two gates
    __builtin_amdgcn_sched_barrier(0);
    r.si[k].template unpack<T>(a);
    r.zi[k].template unpack<T>(b);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const float cnew = fmaf(cact[k][j], sigmoid_f(fmaf(p.alpha, b[j], a[j])), cell[k][j]);
      if (j >= at[k].repeated) ss = fmaf(cnew, cnew, ss);  // unrounded, as in the reference (:136)
      cell[k][j] = cnew;
    }
    const C packed = C::template pack<T>(cell[k]);
    if (at[k].live()) packed.template store_stream<kAnyAlignment>(oc_row + at[k].off);
    packed.template unpack<T>(cell[k]);
  }
  const float inv_cnew = rsqrtf(block_sum(ss, slots_cnew, waves) * p.inv_D + p.eps_state);

  // phase 3: state = gelu(rmsnorm(rounded cell)) * sigmoid(pre_o) (reference :160-190);
  // the output gate is the last load to arrive and is consumed last
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float w[E], b[E], st[E], a[E], g[E];
    vector(ws[k], w, 1.f);
    vector(bs[k], b, 0.f);
#pragma unroll
    for (int j = 0; j < E; ++j) st[j] = gelu<kFastGelu>(fmaf(cell[k][j] * inv_cnew, w[j], b[j]));
    r.so[k].template unpack<T>(a);
    r.zo[k].template unpack<T>(g);
#pragma unroll
    for (int j = 0; j < E; ++j) st[j] *= sigmoid_f(fmaf(p.alpha, g[j], a[j]));
    if (at[k].live()) C::template pack<T>(st).template store_stream<kAnyAlignment>(os_row + at[k].off);
  }
}

// Rows of up to 8192 elements, one chunk of 8 per lane, with the requests of a row issued in stages.  A CU accepts vector-memory requests only as fast as HBM answers them: a wave
// that asks for its nine chunks at once sits in the ninth request for microseconds, long after the first chunks have
// arrived and with nothing computed, and the younger workgroup of the CU does not get its first request in before
// the older one's last.  Here a wave requests its chunks in the order cell gate z, s; forget gate s, z; previous
// cell; input gate s, z; output gate s, z, at four points of its arithmetic (the best of a sweep over the request
// points at 512 rows of 4096):
//   - the cell gate (2 chunks) at the start, with the cell norm's scale / shift pair right behind it;
//   - the forget gate's s behind the first sum of squares;
//   - the rest of the forget gate, the previous cell and the input gate behind the candidate's GELU, the state
//     norm's pair just ahead of them, and a workgroup barrier that waits for no memory behind them, so that every
//     wave of the row has made these requests before any wave makes the next ones;
//   - the output gate behind the forget gate's part of the cell update; it is consumed last, after the state's GELU.
// Waves that are computing leave the request slots to the others, so both rows of a CU arrive gate by gate and every
// stage's arithmetic runs while the next stage is in flight.  The scale / shift vectors (the same for every row,
// cache resident) are requested where they are needed, not ahead of the row: a wave's requests come back in the order
// they were made.  Both outputs are stored and the previous cell is read with streaming accesses (a step's outputs
// are read by the next launches of the step, but a launch boundary writes them back anyway, and stores that stream
// leave earlier).
//
// kZeroCell: the previous cell is all zeros (the first step of a proposal round) and is not read.
// kAhead: few rows of few waves, where nothing else fills the CU while a stage waits for its round trip: all of the row is
// requested at the start, in the same order (launch_lstm has the rule).  With one z for all gates the chunks of `states`
// go first, so that they are on their way while the index of the embedding arrives.
// kParts: few rows leave most CUs idle while a row's waves share the four SIMDs of one, and there the instructions count
// (about 590 a wave: one row of 2048 / 4096 / 8192 elements takes 3.1 / 4.1 / 6.3 us).  The new cell's norm needs the whole
// row, so each of a row's workgroups (blockIdx.y) does the cell update of all of it; the state behind that norm, two fifths
// of the arithmetic, and the stores it does for four waves' chunks alone, one wave per SIMD.  The workgroups of a row read
// the same bytes, so they belong on one XCD: the hardware deals workgroups round robin over the eight, and blockIdx.x counts
// to a multiple of eight.
template <typename T, bool kFastGelu, bool kSharedZ, bool kZeroCell, RowKind kKind, bool kParts, bool kAhead>
__global__ __launch_bounds__(1024) void sum_lstm_staged_kernel(const LstmStagedParams<kSharedZ, kParts> p) {
  __shared__ float slots_cpre[16];
  __shared__ float slots_cnew[16];
  constexpr int E = Chunk::kElems;
  using C = Chunk;
  using std::integral_constant;
  int64_t row = blockIdx.x, z_id = 0;
  if constexpr (kParts) row = min((int)blockIdx.x, p.rows - 1);
  if constexpr (kAhead && kSharedZ) z_id = z_id_of(p, row);
  if constexpr (kParts)   // all of the workgroup
    if ((int)blockIdx.x >= p.rows) return;
  constexpr bool kAny = kKind == kAnyRow;
  const int waves = ((p.D + 7) / 8 + 63) / 64;   // of the workgroup, as launched
  // whether this wave's chunks are this workgroup's to store
  const bool mine = !kParts || __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) == (int)blockIdx.y;
  // the barriers need every wave, so the lanes behind the last chunk run along on it
  const Place at(threadIdx.x, kKind == kFullWaves ? INT32_MAX : p.D);
  const uint32_t off = at.off;
  auto load = [off](const char *q) { return C::load_stream<kAny>(q + off); };
  const int64_t gate_bytes = (int64_t)p.D * 2;
  const char *s_row = p.states + row * p.s_stride * 2;
  const char *z_row = nullptr;
  if constexpr (!(kAhead && kSharedZ)) z_row = p.z4 + z_row_of<kSharedZ>(p, row) * p.z_stride * 2;
  const char *pc_row = kZeroCell ? s_row : p.prev_cell + row * p.pc_stride * 2;
  char *oc_row = p.out_cell + row * p.out_stride * 2;
  char *os_row = p.out_state + row * p.out_stride * 2;

  C in[9];   // zc sc sf zf pc si zi so zo; with kSharedZ the one z chunk stands for all four, with kZeroCell pc is unused
  // requests chunks kFrom ... kTo - 1 of the list above
  auto request = [&](auto from, auto to) {
    constexpr int kFrom = decltype(from)::value, kTo = decltype(to)::value;
    __builtin_amdgcn_sched_barrier(0);   // neither hoisted above the arithmetic in front nor sunk below what follows
    if constexpr (kFrom <= 0 && 0 < kTo) in[0] = load(z_row + (kSharedZ ? 0 : 3 * gate_bytes));
    if constexpr (kFrom <= 1 && 1 < kTo) in[1] = load(s_row + 3 * gate_bytes);
    if constexpr (kFrom <= 2 && 2 < kTo) in[2] = load(s_row);
    if constexpr (kFrom <= 3 && 3 < kTo && !kSharedZ) in[3] = load(z_row);
    if constexpr (kFrom <= 4 && 4 < kTo && !kZeroCell) in[4] = load(pc_row);
    if constexpr (kFrom <= 5 && 5 < kTo) in[5] = load(s_row + gate_bytes);
    if constexpr (kFrom <= 6 && 6 < kTo && !kSharedZ) in[6] = load(z_row + gate_bytes);
    if constexpr (kFrom <= 7 && 7 < kTo) in[7] = load(s_row + 2 * gate_bytes);
    if constexpr (kFrom <= 8 && 8 < kTo && !kSharedZ) in[8] = load(z_row + 2 * gate_bytes);
    __builtin_amdgcn_sched_barrier(0);
  };
  C ws = C::zero(), bs = C::zero();
  auto request_state_vectors = [&] {
    if (mine) {
      ws = load_scale<T, kAny>(p.w_state, off);
      bs = load_shift<kAny>(p.b_state, off);
    }
  };
  if constexpr (kAhead && kSharedZ) {
    request(integral_constant<int, 1>(), integral_constant<int, 3>());
    asm volatile("" : "+s"(z_id));   // the wait for the index is here
    z_row = p.z4 + (p.z_index ? min(max(z_id, (int64_t)0), (int64_t)p.z_rows - 1) : row) * p.z_stride * 2;
    request(integral_constant<int, 0>(), integral_constant<int, 1>());
  } else {
    request(integral_constant<int, 0>(), integral_constant<int, 2>());
  }
  const C wc = load_scale<T, kAny>(p.w_cell, off), bc = load_shift<kAny>(p.b_cell, off);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (kAhead) {
    request(integral_constant<int, kSharedZ ? 3 : 2>(), integral_constant<int, 7>());
    request_state_vectors();
    if (mine) request(integral_constant<int, 7>(), integral_constant<int, 9>());
    __builtin_amdgcn_sched_barrier(0);
  }

  // phase 1: pre_c and its sum of squares (reference :65-82)
  float cact[E], a[E], b[E], c[E];
  float ss = 0.f;
  in[1].template unpack<T>(a);
  in[0].template unpack<T>(b);
#pragma unroll
  for (int j = 0; j < E; ++j) {
    cact[j] = fmaf(p.alpha, b[j], a[j]);
    if (!kAny || j >= at.repeated) ss = fmaf(cact[j], cact[j], ss);
  }
  if constexpr (!kAhead) request(integral_constant<int, 2>(), integral_constant<int, 3>());
  const float inv_cpre = rsqrtf(block_sum(kKind != kRagged || at.live() ? ss : 0.f, slots_cpre, waves) * p.inv_D + p.eps_cell);
  {
    float w[E], sh[E];
    wc.template unpack<T>(w);
    bc.template unpack<T>(sh);
#pragma unroll
    for (int j = 0; j < E; ++j) cact[j] = gelu<kFastGelu>(fmaf(cact[j] * inv_cpre, w[j], sh[j]));
  }
  if constexpr (!kAhead) {
    request_state_vectors();
    request(integral_constant<int, 3>(), integral_constant<int, 7>());
    __builtin_amdgcn_s_barrier();   // waits for no memory: only keeps the row's waves in step at their largest group of requests
  }
  __builtin_amdgcn_sched_barrier(0);

  // phase 2: cell update; write out_cell (reference :104-140)
  float cell[E];
  in[2].template unpack<T>(a);
  (kSharedZ ? in[0] : in[3]).template unpack<T>(b);
  (kZeroCell ? C::zero() : in[4]).template unpack<T>(c);
#pragma unroll
  for (int j = 0; j < E; ++j) cell[j] = sigmoid_f(fmaf(p.alpha, b[j], a[j])) * c[j];
  __builtin_amdgcn_sched_barrier(0);   // the forget gate's part stays ahead of the wait for the input gate
  in[5].template unpack<T>(a);
  (kSharedZ ? in[0] : in[6]).template unpack<T>(b);
  ss = 0.f;
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const float cnew = fmaf(cact[j], sigmoid_f(fmaf(p.alpha, b[j], a[j])), cell[j]);
    if (!kAny || j >= at.repeated) ss = fmaf(cnew, cnew, ss);  // unrounded, as in the reference (:136)
    cell[j] = cnew;
  }
  {
    const C packed = C::template pack<T>(cell);
    if (mine && (kKind == kFullWaves || at.live())) packed.template store_stream<kAny>(oc_row + off);
    packed.template unpack<T>(cell);   // the state phase sees the rounded cell (:163,174)
  }
  if constexpr (!kAhead)
    if (mine) request(integral_constant<int, 7>(), integral_constant<int, 9>());
  const float inv_cnew = rsqrtf(block_sum(kKind != kRagged || at.live() ? ss : 0.f, slots_cnew, waves) * p.inv_D + p.eps_state);
  if (!mine) return;   // behind the last barrier

  // phase 3: state = gelu(rmsnorm(rounded cell)) * sigmoid(pre_o) (reference :160-190)
  float st[E];
  {
    float w[E], sh[E];
    ws.template unpack<T>(w);
    bs.template unpack<T>(sh);
#pragma unroll
    for (int j = 0; j < E; ++j) st[j] = gelu<kFastGelu>(fmaf(cell[j] * inv_cnew, w[j], sh[j]));
  }
  __builtin_amdgcn_sched_barrier(0);   // the GELU above runs while the output gate is still on its way
  in[7].template unpack<T>(a);
  (kSharedZ ? in[0] : in[8]).template unpack<T>(b);
#pragma unroll
  for (int j = 0; j < E; ++j) st[j] *= sigmoid_f(fmaf(p.alpha, b[j], a[j]));
  if (kKind == kFullWaves || at.live()) C::template pack<T>(st).template store_stream<kAny>(os_row + off);
}

// Any D, any alignment: element-wise, three passes like the reference's scalar
// kernel (sum_lstm.cu:193-291).
constexpr int kScalarLanes = 256;
struct LstmScalarParams : LstmCall {
  int z_gate_stride;   // elements between two gates of z4: 0 when they share one
};
template <typename T, bool kFastGelu>
__global__ __launch_bounds__(kScalarLanes) void sum_lstm_scalar_kernel(const LstmScalarParams p) {
  __shared__ float slots_cpre[16];
  __shared__ float slots_cnew[16];
  const int D = p.D;
  const int64_t row = blockIdx.x;
  const uint16_t *s = (const uint16_t *)p.states + row * p.s_stride;
  const uint16_t *z = (const uint16_t *)p.z4 + z_row_of<true>(p, row) * p.z_stride;
  const uint16_t *pc = (const uint16_t *)p.prev_cell + row * p.pc_stride;
  uint16_t *oc = (uint16_t *)p.out_cell + row * p.out_stride;
  uint16_t *os = (uint16_t *)p.out_state + row * p.out_stride;
  const uint16_t *wc = (const uint16_t *)p.w_cell, *bc = (const uint16_t *)p.b_cell;
  const uint16_t *ws = (const uint16_t *)p.w_state, *bs = (const uint16_t *)p.b_state;

  float ss = 0.f;
  for (int j = threadIdx.x; j < D; j += kScalarLanes) {
    const float c = T::lo(s[3 * (int64_t)D + j]) + p.alpha * T::lo(z[3 * (int64_t)p.z_gate_stride + j]);
    ss += c * c;
  }
  const float inv_cpre = rsqrtf(block_sum(ss, slots_cpre, kScalarLanes / 64) * p.inv_D + p.eps_cell);

  ss = 0.f;
  for (int j = threadIdx.x; j < D; j += kScalarLanes) {
    const float pre_f = T::lo(s[j]) + p.alpha * T::lo(z[j]);
    const float pre_i = T::lo(s[(int64_t)D + j]) + p.alpha * T::lo(z[(int64_t)p.z_gate_stride + j]);
    const float cpre = T::lo(s[3 * (int64_t)D + j]) + p.alpha * T::lo(z[3 * (int64_t)p.z_gate_stride + j]);
    float cn = cpre * inv_cpre;
    if (wc) cn *= T::lo(wc[j]);
    if (bc) cn += T::lo(bc[j]);
    const float cnew = (p.prev_cell ? T::lo(pc[j]) : 0.f) * sigmoid_f(pre_f) + gelu<kFastGelu>(cn) * sigmoid_f(pre_i);
    ss += cnew * cnew;
    oc[j] = (uint16_t)T::round_bits(cnew);
  }
  const float inv_cnew = rsqrtf(block_sum(ss, slots_cnew, kScalarLanes / 64) * p.inv_D + p.eps_state);

  // each thread re-reads only the out_cell elements it wrote itself
  for (int j = threadIdx.x; j < D; j += kScalarLanes) {
    float cn = T::lo(oc[j]) * inv_cnew;
    if (ws) cn *= T::lo(ws[j]);
    if (bs) cn += T::lo(bs[j]);
    const float pre_o = T::lo(s[2 * (int64_t)D + j]) + p.alpha * T::lo(z[2 * (int64_t)p.z_gate_stride + j]);
    os[j] = (uint16_t)T::round_bits(gelu<kFastGelu>(cn) * sigmoid_f(pre_o));
  }
}

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Whether an output shares memory with a gate or the previous cell: `columns` elements of each of `rows` rows, `stride`
// elements apart, looked at as whole ranges.
static bool in_place(const LstmCall &p, int64_t rows, bool shared_z) {
  const auto overlaps = [&](const char *out, const char *in, int64_t in_rows, int64_t stride, int64_t columns) {
    const uintptr_t o = (uintptr_t)out, i = (uintptr_t)in;
    return in && o < i + (uintptr_t)((in_rows - 1) * stride + columns) * 2 &&
           i < o + (uintptr_t)((rows - 1) * p.out_stride + p.D) * 2;
  };
  const int64_t gates = 4 * (int64_t)p.D;
  for (const char *out : {p.out_state, p.out_cell})
    if (overlaps(out, p.states, rows, p.s_stride, gates) || overlaps(out, p.prev_cell, rows, p.pc_stride, p.D) ||
        overlaps(out, p.z4, p.z_index ? p.z_rows : rows, p.z_stride, shared_z ? p.D : gates))
      return true;
  return false;
}

template <typename T, bool kFastGelu, bool kSharedZ>
static void launch_lstm(const LstmCall &p, int64_t rows, hipStream_t s) {
  const bool multi = rows > 1;
  // The vector kernels' arguments are 32 bits wide.  Rows 2^32 elements and more apart (8 GiB, so there are few) are launched
  // one by one, where no pitch counts; a table of embeddings with such rows is the element-wise kernel's.
  const auto fits = [](int64_t v) { return v <= (int64_t)UINT32_MAX; };
  if (multi && !(fits(p.s_stride) && fits(p.pc_stride) && fits(p.out_stride) && (p.z_index || fits(p.z_stride)))) {
    for (int64_t r = 0; r < rows; ++r) {
      LstmCall one = p;
      one.out_state += r * p.out_stride * 2;
      one.out_cell += r * p.out_stride * 2;
      one.states += r * p.s_stride * 2;
      if (p.prev_cell) one.prev_cell += r * p.pc_stride * 2;
      if (p.z_index) one.z_index += r;
      else one.z4 += r * p.z_stride * 2;
      launch_lstm<T, kFastGelu, kSharedZ>(one, 1, s);
    }
    return;
  }
  const bool aligned = p.D % 8 == 0 &&
                       (!multi || (p.s_stride % 8 == 0 && p.z_stride % 8 == 0 && p.pc_stride % 8 == 0 &&
                                   p.out_stride % 8 == 0)) &&
                       (!p.z_index || p.z_stride % 8 == 0) &&
                       aligned16(p.states) && aligned16(p.z4) && aligned16(p.prev_cell) &&   /* null counts as aligned */
                       aligned16(p.out_state) && aligned16(p.out_cell) && aligned16(p.w_cell) &&
                       aligned16(p.b_cell) && aligned16(p.w_state) && aligned16(p.b_state);
  const int chunks = (p.D + 7) / 8;
  const int lanes = (chunks + 63) & ~63;
  dim3 grid((unsigned)rows);
  // One chunk per lane up to 1024 lanes (512 rows of 5120 / 6144 / 8192 elements: 12.0 / 13.9 / 17.5 us against 17.6 /
  // 19.9 / 22.5 us with two chunks per lane in the other kernel; without scale and shift 512 rows of 4096 / 8192: 9.6 /
  // 17.3 us against 11.0 / 24.1 us).  Rows that are not 16-byte aligned take the same kernels with accesses at any
  // alignment, which cost 6 to 35 % over aligned ones (300 rows of 1536: 5.3 us aligned, 5.8 us 4-byte and 6.4 us 2-byte
  // aligned) and are 3 to 5 times faster than element by element (23 us; 300 rows of 4096: 10.9 against 58 us).  Up to 256
  // elements the element-wise kernel gives every element a lane of its own where one to four half-idle waves would do a
  // row's whole arithmetic in chunks (us element by element / in chunks, rows x elements, without vectors: 64 x 128 2.67 /
  // 3.30, 512 x 128 3.01 / 3.87, 64 x 256 2.77 / 3.27, 4096 x 256 8.7 / 9.5; with all of them 512 x 128 3.31 / 3.88, 64 x
  // 256 3.07 / 3.24); with all vectors and more than 256 rows it is chunks from 129 on (300 x 136 level, 512 x 160 7 % and
  // 2048 x 256 8 % faster).  From 257 on chunks are faster at every row count (64 x 257 by 10 to 23 %, 64 x 513 by 21 to 35).
#define ARCTIC_LSTM_STAGED_LAUNCH(ZERO, KIND, PARTS, AHEAD, PARAMS) \
  launch(sum_lstm_staged_kernel<T, kFastGelu, kSharedZ, ZERO, KIND, PARTS, AHEAD>, grid, lanes, s, PARAMS)
#define ARCTIC_LSTM_STAGED_AS(ZERO, KIND)                                                                     \
  do {                                                                                                        \
    if (in_parts && kSharedZ && parts_ahead) ARCTIC_LSTM_STAGED_LAUNCH(ZERO, KIND, true, kSharedZ, of_parts); \
    else if (in_parts) ARCTIC_LSTM_STAGED_LAUNCH(ZERO, KIND, true, false, of_parts);                          \
    else if (ahead) ARCTIC_LSTM_STAGED_LAUNCH(ZERO, KIND, false, true, compact);                              \
    else ARCTIC_LSTM_STAGED_LAUNCH(ZERO, KIND, false, false, compact);                                        \
  } while (0)
#define ARCTIC_LSTM_STAGED(KIND)                          \
  do {                                                    \
    if (p.prev_cell) ARCTIC_LSTM_STAGED_AS(false, KIND);  \
    else ARCTIC_LSTM_STAGED_AS(true, KIND);               \
  } while (0)
  const bool all_vectors = p.w_cell && p.b_cell && p.w_state && p.b_state;
  const bool narrow = !aligned && p.D <= (all_vectors && rows > 256 ? 128 : 256);
  // A call that updates a tensor in place relies on every element being read before it is written.  In a width that is no
  // multiple of 8 two lanes, at some widths (513, 1537) of two waves, read the last elements of a row and both store them,
  // and nothing orders the one's load before the other's store: such a call goes element by element.  Aligned rows that
  // lack a vector are requested together, since the stages read the output gate behind the first store.
  const bool aliased = (p.D % 8 || !all_vectors) && in_place(p, rows, kSharedZ);
  const bool element_wise = narrow || (aliased && p.D % 8) || !fits(p.z_rows) || (p.z_index && !fits(p.z_stride)) || chunks > 2 * 1024;
  LstmParamsOf<kSharedZ> compact;
  static_cast<LstmParams<uint32_t> &>(compact) = {
      p.out_state, p.out_cell, p.states, p.z4, p.prev_cell, p.w_cell, p.b_cell, p.w_state, p.b_state, (uint32_t)p.s_stride,
      (uint32_t)p.z_stride, (uint32_t)p.pc_stride, (uint32_t)p.out_stride, (uint32_t)p.z_rows, p.D, p.inv_D, p.alpha,
      p.eps_cell, p.eps_state};
  if constexpr (kSharedZ) compact.z_index = p.z_index;
  // At most four waves per row and few rows: everything is requested ahead, since a CU with a row or two of one to four waves
  // takes the requests as they come, and a stage that waits for its round trip has nobody to leave the CU to.  Us per call in a
  // graph, in stages / ahead: 7 x 1024 3.25 / 2.93, 64 x 2048 4.15 / 3.58, 256 x 1537 5.48 / 4.53, 512 x 512 4.14 / 3.48,
  // 1000 x 512 4.57 / 4.29, 512 x 1500 6.29 / 6.00, embedded 256 x 2048 4.55 / 4.01; behind the lines below 2000 x 512 5.27 /
  // 5.41, 700 x 1024 5.46 / 5.77, one z for all gates 400 x 2048 5.38 / 5.56, and with more waves per row 512 x 4096 9.09 / 9.99.
  const int64_t ahead_rows = chunks <= 64 ? 1024 : chunks > 256 ? 0 : kSharedZ && aligned && chunks > 192 ? 256 : 512;
  const bool ahead = rows <= ahead_rows;
  // Rows of up to 2048 elements that lack a vector: at most four waves per row, whose loads are few enough to be
  // requested together.  Aligned ones, us per call in a graph, in stages (ones and zeros read in place of an absent vector) / together:
  // 64 x 256 without vectors 4.0 / 3.2, 512 x 512 4.2 / 3.3, 300 x 2048 5.6 / 4.8, 512 x 512 with the scales alone 4.1 / 3.4;
  // from 513 elements and 513 rows on the stages are faster (2048 x 1024 8.8 / 9.4), but for one z for all gates (8.4 / 7.7).
  // Rows at any alignment do it without any vector, or with one wave per row: 300 x 1537 without 5.89 / 5.34, 64 x 513 3.57 /
  // 3.26, 1500 x 257 5.58 / 4.88, with one z for all gates 1500 x 1537 11.1 / 10.0; with the scales alone 300 x 300 3.41 /
  // 3.33, but 300 x 769 4.62 / 4.84 (without any vector 4.70 / 4.59, and without a previous cell either 4.54 / 4.63).
  // Where rows are requested ahead (above) that is as good for the ones with some vectors: 64 x 1024 3.47 / 3.36, 256 x 512 3.49
  // / 3.42; calls that update a tensor in place stay here.
  const bool no_vector = !p.w_cell && !p.b_cell && !p.w_state && !p.b_state;
  const bool together = !all_vectors && chunks <= 256 && (chunks <= 64 || ((aligned || no_vector) && (rows <= 512 || kSharedZ))) &&
                        (no_vector || aliased || !ahead);
#define ARCTIC_LSTM_VEC_LAUNCH(K, ANY, BARE) \
  launch(sum_lstm_vec_kernel<T, K, kFastGelu, kSharedZ, ANY, BARE>, grid, threads, s, compact)
#define ARCTIC_LSTM_VEC(K, ANY)                                       \
  do {                                                                \
    const int threads = ((chunks + (K) - 1) / (K) + 63) & ~63;        \
    if (no_vector) ARCTIC_LSTM_VEC_LAUNCH(K, ANY, true);              \
    else ARCTIC_LSTM_VEC_LAUNCH(K, ANY, false);                       \
  } while (0)
  if (element_wise) {
    launch(sum_lstm_scalar_kernel<T, kFastGelu>, grid, kScalarLanes, s, LstmScalarParams{p, kSharedZ ? 0 : p.D});
  } else if (together && aligned) {
    ARCTIC_LSTM_VEC(1, false);
  } else if (together) {
    ARCTIC_LSTM_VEC(1, true);
  } else if (aliased && aligned) {
    ARCTIC_LSTM_VEC(2, false);
  } else if (chunks <= 1024) {
    // Few rows of more than 2048 elements: a workgroup per four waves of a row, as long as every workgroup has a CU of its
    // own.  Us per call in a graph, one workgroup per row / in parts: 7 x 4096 4.14 / 3.87, 3 x 8192 6.30 / 5.50, 45 x 5120
    // 6.16 / 5.40, 64 x 8192 7.71 / 7.11, 128 x 4096 5.41 / 5.18; with two workgroups on a CU 85 x 5120 6.39 / 8.01, and
    // with a last part of less than four waves it is level from 200 workgroups on (128 x 2880 5.16 / 5.23).  A call that
    // updates a tensor in place would read in one workgroup what another one has written.
    const int parts = (lanes + 255) / 256;
    const int64_t rows_up = (rows + 7) & ~(int64_t)7;
    const bool in_parts = parts > 1 && rows_up * parts <= (lanes % 256 ? 224 : 256) && !in_place(p, rows, kSharedZ);
    // One z for all gates leaves few enough requests to make them ahead (embedded, in stages / ahead: 7 x 2880 4.07 / 3.90, 64 x
    // 2880 4.19 / 4.11, 7, 10, 16, 24, 32 and 64 x 4096 4.17 / 4.00, 4.17 / 3.97, 4.13 / 4.00, 4.21 / 4.02, 4.16 / 4.06 and 4.68 /
    // 4.63, where it is level).  Rows at any alignment are not faster for it: pitched by 1, 8 x 3600 3.9 to 8 % slower, 8 x 4096 7 to
    // 8 %, 8 x 2880 1 to 6 %, odd widths between 5 % faster and 4 % slower.
    const bool parts_ahead = aligned && (lanes <= 384 || (lanes <= 512 && rows <= 16));
    LstmPartsParams<kSharedZ> of_parts;
    if (in_parts) {
      static_cast<LstmParamsOf<kSharedZ> &>(of_parts) = compact;
      of_parts.rows = (int)rows;
      grid = dim3((unsigned)rows_up, (unsigned)parts);
    }
    if (!aligned || !all_vectors) ARCTIC_LSTM_STAGED(kAnyRow);
    else if (lanes != chunks) ARCTIC_LSTM_STAGED(kRagged);
    else ARCTIC_LSTM_STAGED(kFullWaves);
  } else if (aligned) {
    ARCTIC_LSTM_VEC(2, false);
  } else {
    ARCTIC_LSTM_VEC(2, true);
  }
#undef ARCTIC_LSTM_VEC
#undef ARCTIC_LSTM_VEC_LAUNCH
#undef ARCTIC_LSTM_STAGED
#undef ARCTIC_LSTM_STAGED_AS
#undef ARCTIC_LSTM_STAGED_LAUNCH
}

}  // namespace arctic

using namespace arctic;

static int sum_lstm_entry(const char *fn, bool shared_z, void *out_state, void *out_cell, const void *states,
                          const void *z, const int64_t *z_index, int64_t z_rows, const void *prev_cell, const void *w_cell, const void *b_cell,
                          const void *w_state, const void *b_state, int64_t rows, int D, int64_t s_stride,
                          int64_t z_stride, int64_t pc_stride, int64_t out_stride, float alpha, float eps_cell,
                          float eps_state, int fast_gelu, int dtype, void *stream) {
  if (dtype != ARCTIC_DTYPE_F16 && dtype != ARCTIC_DTYPE_BF16)
    return fail(ARCTIC_ERR_UNSUPPORTED, "%s: only fp16 and bf16 are supported.", fn);
  if (D <= 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: last dim of states must be 4*D_gate", fn);
  if (rows < 0 || rows > 0x7fffffffLL) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: bad row count", fn);
  if (rows == 0) return ARCTIC_OK;
  if (!out_state || !out_cell || !states || !z)   // prev_cell may be null: a cell of zeros
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null tensor pointer", fn);
  if (z_index && z_rows <= 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: the embedding table has no rows", fn);
  if (D > (1 << 28)) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: D_gate beyond 2^28", fn);
  if (!pitch_ok(s_stride, rows, 2) || !pitch_ok(z_stride, z_index ? z_rows : rows, 2) ||
      !pitch_ok(pc_stride, rows, 2) || !pitch_ok(out_stride, rows, 2))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: row pitch out of range", fn);
  LstmCall p;
  p.z_index = z_index;
  p.z_rows = z_rows;
  p.out_state = (char *)out_state;
  p.out_cell = (char *)out_cell;
  p.states = (const char *)states;
  p.z4 = (const char *)z;
  p.prev_cell = (const char *)prev_cell;
  p.w_cell = (const char *)w_cell;
  p.b_cell = (const char *)b_cell;
  p.w_state = (const char *)w_state;
  p.b_state = (const char *)b_state;
  p.s_stride = s_stride;
  p.z_stride = z_stride;
  p.pc_stride = prev_cell ? pc_stride : 0;
  p.out_stride = out_stride;
  p.D = D;
  p.inv_D = 1.0f / (float)D;
  p.alpha = alpha;
  p.eps_cell = eps_cell;
  p.eps_state = eps_state;
  hipStream_t s = (hipStream_t)stream;
#define ARCTIC_LSTM_DISPATCH(TYPE)                                        \
  do {                                                                    \
    if (shared_z) {                                                       \
      if (fast_gelu) launch_lstm<TYPE, true, true>(p, rows, s);           \
      else launch_lstm<TYPE, false, true>(p, rows, s);                    \
    } else {                                                              \
      if (fast_gelu) launch_lstm<TYPE, true, false>(p, rows, s);          \
      else launch_lstm<TYPE, false, false>(p, rows, s);                   \
    }                                                                     \
  } while (0)
  if (dtype == ARCTIC_DTYPE_BF16) ARCTIC_LSTM_DISPATCH(BF16);
  else ARCTIC_LSTM_DISPATCH(F16);
#undef ARCTIC_LSTM_DISPATCH
  return check_launch(fn);
}

extern "C" int arctic_sum_lstm(void *out_state, void *out_cell, const void *states, const void *z4,
                               const void *prev_cell, const void *w_cell, const void *b_cell,
                               const void *w_state, const void *b_state, int64_t rows, int D,
                               int64_t s_stride, int64_t z_stride, int64_t pc_stride, int64_t out_stride,
                               float alpha, float eps_cell, float eps_state, int fast_gelu, int dtype,
                               void *stream) {
  return sum_lstm_entry("sum_lstm", false, out_state, out_cell, states, z4, nullptr, 0, prev_cell, w_cell, b_cell, w_state,
                        b_state, rows, D, s_stride, z_stride, pc_stride, out_stride, alpha, eps_cell, eps_state,
                        fast_gelu, dtype, stream);
}

extern "C" int arctic_sum_lstm_shared_z(void *out_state, void *out_cell, const void *states, const void *z,
                                        const void *prev_cell, const void *w_cell, const void *b_cell,
                                        const void *w_state, const void *b_state, int64_t rows, int D,
                                        int64_t s_stride, int64_t z_stride, int64_t pc_stride,
                                        int64_t out_stride, float alpha, float eps_cell, float eps_state,
                                        int fast_gelu, int dtype, void *stream) {
  return sum_lstm_entry("sum_lstm_shared_z", true, out_state, out_cell, states, z, nullptr, 0, prev_cell, w_cell, b_cell,
                        w_state, b_state, rows, D, s_stride, z_stride, pc_stride, out_stride, alpha, eps_cell,
                        eps_state, fast_gelu, dtype, stream);
}

extern "C" int arctic_sum_lstm_embedded(void *out_state, void *out_cell, const void *states, const void *emb_table,
                                        const int64_t *token_ids, const void *prev_cell, const void *w_cell,
                                        const void *b_cell, const void *w_state, const void *b_state, int64_t rows,
                                        int D, int64_t s_stride, int64_t emb_stride, int64_t pc_stride,
                                        int64_t out_stride, int64_t num_embeddings, float alpha, float eps_cell,
                                        float eps_state, int fast_gelu, int dtype, void *stream) {
  const char *fn = "sum_lstm_embedded";
  if (rows > 0 && !token_ids) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null token ids", fn);
  return sum_lstm_entry(fn, true, out_state, out_cell, states, emb_table, token_ids, num_embeddings, prev_cell, w_cell,
                        b_cell, w_state, b_state, rows, D, s_stride, emb_stride, pc_stride, out_stride, alpha, eps_cell,
                        eps_state, fast_gelu, dtype, stream);
}
