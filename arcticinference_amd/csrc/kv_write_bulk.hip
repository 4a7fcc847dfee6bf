// SwiftKV bulk KV-cache write for gfx950.
//
// Replaces reshape_and_cache_flash_bulk (host launcher and kernel,
// csrc/custom_ops/reshape_and_cache_flash_bulk.cu:12-144 in the reference).
//
// Work decomposition
// ------------------
// One workgroup owns one token and a run of consecutive layers.  The token's
// slot is looked up once; a prologue turns (slot, layer, K|V) into a table of
// row descriptors in LDS - destination address of the token's row in that
// layer's cache and the fp64 reciprocal of that layer's scale - with one lane per
// row, so the per-layer pointer and scale reads are issued together instead of
// one dependent pair per layer.  The main loop then streams the token's source
// rows: every lane moves 16 bytes per access (8 bf16/fp16 or 4 fp32 elements),
// consecutive lanes cover consecutive addresses along head_size, and the cache
// row is written with 16-byte (copy) or 8-byte (fp8, 8 codes) stores.  Source
// and destination are each touched exactly once, so both use streaming
// (non-temporal) accesses.  Stores written through the L2 instead end in the
// 256 MB memory-side cache and leave the launch sooner (5003 tokens x 33 layers
// of 3 x 96 to fp8, launch behind launch: 58 us against 70), but the work behind
// the launch then waits for those lines to reach HBM.  What a launch adds to a
// step that goes on to read 1.05 GB of weights, streaming / through: that launch
// 72 / 91 us, 1024 x 33 of it 16.2 / 22.9, 512 x 40 of 8 x 128 24.8 / 33.7,
// 1024 x 40 48.5 / 59.2, 1024 x 16 as they are 26.8 / 37.7.
//
// The four per-layer pointer tables travel in the kernel-argument segment, so a
// call uploads nothing and can be recorded into a HIP graph.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "fp8_convert.hpp"

namespace arctic {

constexpr int kScalarThreads = 256;
constexpr int kLayersPerLaunch = 64;  // 4 tables x 64 pointers = 2 KiB of kernel arguments
// Launches of up to this many layers take tables of that size where the launch's own cost counts (launch_vec_shape).
constexpr int kFewLayers = 16;

template <int kLayers>
struct LayerTables {
  const void *key_cache[kLayers];
  const void *value_cache[kLayers];
  const float *k_scale[kLayers];
  const float *v_scale[kLayers];
};

struct BulkParams {
  const char *keys;    // already offset to the first layer of this launch
  const char *values;
  const int64_t *slot_mapping;
  int64_t key_stride_bytes;
  int64_t value_stride_bytes;
  int64_t block_stride;  // elements
  int64_t num_slots;     // slots at or beyond this move nothing
  int num_layers;        // layers in this launch
  int layers_per_group;  // consecutive layers owned by one workgroup
  int groups_per_token;
  int n;                 // num_heads * head_size
  int block_size;
  int chunks_per_row;    // 16-byte source chunks per (token, layer) row
  int chunk_shift;       // log2(chunks_per_row) or -1
  // The places of a chunk, a slot and a workgroup by products: general divisions stand between the slot's arrival and the
  // first store, and in rows that are no power of two long one per chunk (us per call in a graph, before / after: 5 tokens
  // x 16 layers of 8 x 128 to fp8 3.08 / 2.97, 64 x 33 of 3 x 96 4.52 / 4.11, 1024 x 33 15.1 / 14.4).
  Divisor by_chunks;     // chunks_per_row
  Divisor by_block;      // block_size
  Divisor by_groups;     // groups_per_token
};

struct BulkSelectParams : BulkParams {
  // select variants: token t's source rows are also copied, unconverted, to the rows j of keys_out / values_out with
  // indices[j] == t.  With a row map (kSelectByRowMap) that is row row_map[t] of keys_out /
  // values_out (already offset to the first layer of this launch); a negative row or one >= num_out_rows = none
  const int64_t *row_map;
  char *keys_out;
  char *values_out;
  int64_t out_key_stride_bytes;
  int64_t out_value_stride_bytes;
  int64_t num_out_rows;
  // The first index_blocks workgroups serve the index list itself, one output row per lane: output row j whose
  // index the row map does not credit to j (a repeated index, or a source row at or beyond num_tokens) is copied
  // straight from source row indices[j], so the output equals index_select for every index in [0, num_src_rows).
  // A handful of workgroups, first in the grid so that their two dependent lookups overlap the token workgroups'
  // streaming instead of trailing it.  indices == nullptr: no such workgroups are launched.
  const void *indices;
  int64_t num_tokens;
  int64_t num_src_rows;
  unsigned index_blocks;
  int index_is_64;
  int select_mode;   // kSelectNone / kSelectByRowMap / kSelectByScan (the vector kernels take it as a template argument)
};

// How a launch finds the output rows of a token: not at all, through the inverse of the index list that the caller
// built beforehand, or by scanning the index list itself (short lists: one or a few loads per lane, no launch and
// no workspace for the inverse).
enum : int { kSelectNone = 0, kSelectByRowMap = 1, kSelectByScan = 2 };

template <int kSelect>
struct ParamsFor { using type = BulkSelectParams; };
template <>
struct ParamsFor<kSelectNone> { using type = BulkParams; };
template <int kSelect>
using BulkParamsOf = typename ParamsFor<kSelect>::type;

struct __align__(16) RowDesc {
  char *dst;    // first byte of this token's row in the layer's K or V cache
  double inv;   // RN64(1 / scale); unused by the copy path
};

// ---- element-type plumbing ---------------------------------------------------
struct SrcBF16 {
  static constexpr int kElemsPerChunk = 8;
  static constexpr int kBytes = 2;
  __device__ static __forceinline__ void to_float(const uint4 &v, float (&f)[8]) { unpack8<BF16>(v, f); }
};
struct SrcF16 {
  static constexpr int kElemsPerChunk = 8;
  static constexpr int kBytes = 2;
  __device__ static __forceinline__ void to_float(const uint4 &v, float (&f)[8]) { unpack8<F16>(v, f); }
};
struct SrcF32 {
  static constexpr int kElemsPerChunk = 4;
  static constexpr int kBytes = 4;
};

struct Copy {};  // ARCTIC_KV_AUTO

template <typename F8>
__device__ __forceinline__ void quantize_store(char *dst, const float (&f)[8], double inv) {
  uint2 out;
  out.x = encode4<F8>(div_by_scale(f[0], inv), div_by_scale(f[1], inv),
                      div_by_scale(f[2], inv), div_by_scale(f[3], inv));
  out.y = encode4<F8>(div_by_scale(f[4], inv), div_by_scale(f[5], inv),
                      div_by_scale(f[6], inv), div_by_scale(f[7], inv));
  store8_stream(dst, out);
}

// One 16-byte source chunk -> cache.  `col` is the chunk's index inside its row.
template <typename Src, typename Dst>
__device__ __forceinline__ void emit_chunk(const uint4 &v, const RowDesc &d, int col) {
  if constexpr (std::is_same<Dst, Copy>::value) {
    store16_stream(d.dst + (int64_t)col * 16, v);
  } else if constexpr (Src::kElemsPerChunk == 8) {
    float f[8];
    Src::to_float(v, f);
    quantize_store<Dst>(d.dst + (int64_t)col * 8, f, d.inv);
  } else {
    const uint32_t w = encode4<Dst>(div_by_scale(__uint_as_float(v.x), d.inv),
                                    div_by_scale(__uint_as_float(v.y), d.inv),
                                    div_by_scale(__uint_as_float(v.z), d.inv),
                                    div_by_scale(__uint_as_float(v.w), d.inv));
    store4_stream(d.dst + (int64_t)col * 4, w);
  }
}

// Which source row output row j wants, or -1 when the token workgroups already copy it or the index lies outside
// the source.  By row map: the token's workgroup serves the one output row the map credits the token with.  By scan:
// it serves every output row that names the token, so only source rows beyond the slot mapping are left.
template <int kSelect>
__device__ __forceinline__ int64_t leftover_source_row(const BulkSelectParams &p, int64_t j) {
  const int64_t t = p.index_is_64 ? ((const int64_t *)p.indices)[j] : (int64_t)((const int32_t *)p.indices)[j];
  if (t < 0 || t >= p.num_src_rows) return -1;
  if (t < p.num_tokens && (kSelect == kSelectByScan || p.row_map[t] == j)) return -1;
  return t;
}

// Index workgroup `b`: its lanes look at output rows b * kThreads ... (one each); almost always none of them is
// left over (SwiftKV selects each token once) and the workgroup is done after two dependent lookups.  The rows that
// are left over are listed in LDS and copied by the whole workgroup, all layers of the launch, one row after the other.
template <int kThreads, int kSelect>
__device__ __forceinline__ int list_leftover_rows(const BulkSelectParams &p, unsigned b, int64_t (&todo_j)[kThreads],
                                                  int64_t (&todo_t)[kThreads], int &count) {
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  const int64_t j = (int64_t)b * kThreads + threadIdx.x;
  if (j < p.num_out_rows) {
    const int64_t t = leftover_source_row<kSelect>(p, j);
    if (t >= 0) {
      const int k = atomicAdd(&count, 1);
      todo_j[k] = j;
      todo_t[k] = t;
    }
  }
  __syncthreads();
  return count;
}

template <typename Src, bool kPow2, int kBulkThreads, int kSelect>
__device__ __forceinline__ void select_leftover_rows(const BulkSelectParams &p, unsigned b) {
  __shared__ int64_t todo_j[kBulkThreads], todo_t[kBulkThreads];
  __shared__ int count;
  const int n = list_leftover_rows<kBulkThreads, kSelect>(p, b, todo_j, todo_t, count);
  const int cpr = p.chunks_per_row;
  const int total = 2 * p.num_layers * cpr;
  for (int e = 0; e < n; ++e) {
    const int64_t j = todo_j[e], t = todo_t[e];
    const char *ksrc = p.keys + t * p.key_stride_bytes, *vsrc = p.values + t * p.value_stride_bytes;
    char *kout = p.keys_out + j * p.out_key_stride_bytes, *vout = p.values_out + j * p.out_value_stride_bytes;
    for (int c = threadIdx.x; c < total; c += kBulkThreads) {
      int r, col;
      if constexpr (kPow2) {
        r = c >> p.chunk_shift;
        col = c & (cpr - 1);
      } else {
        r = c / cpr;
        col = c - r * cpr;
      }
      const int64_t off = ((int64_t)(r >> 1) * cpr + col) * 16;
      store16_stream(((r & 1) ? vout : kout) + off, load16_stream(((r & 1) ? vsrc : ksrc) + off));
    }
  }
}

// kBulkThreads x kUnroll 16-byte chunks form one batch of a workgroup.  Three shapes are built, all with batches
// of 1024 chunks: 1024 x 1 (launches of more than 8192 tokens, or 4096 of rows that are no power of two long: a workgroup
// moves up to five batches), 512 x 2 (launches of more than 8192 tokens that select rows as well) and 256 x 4 (everything
// else: up to two batches per workgroup, rounded up to whole layers, and up to five where more than 8192 tokens of rows
// that are no power of two long select).
template <typename Src, typename Dst, bool kPow2, int kBulkThreads, int kUnroll, int kSelect, bool kWholeAhead, typename Params,
          typename Tables>
__device__ __forceinline__ void bulk_item(const Params &p, const Tables &tab, unsigned block) {
  constexpr bool kCopy = std::is_same<Dst, Copy>::value;
  constexpr int kDstElemBytes = kCopy ? Src::kBytes : 1;

  __shared__ RowDesc rows[2 * kLayersPerLaunch];

  if constexpr (kSelect) {
    if (block < p.index_blocks) {  // uniform over the workgroup, before any barrier
      select_leftover_rows<Src, kPow2, kBulkThreads, kSelect>(p, block);
      return;
    }
    block -= p.index_blocks;
  }
  const int64_t token = p.by_groups.quotient(block);
  const int group = block - (unsigned)token * (unsigned)p.groups_per_token;
  const int layer0 = group * p.layers_per_group;
  const int nlayers = min(p.layers_per_group, p.num_layers - layer0);

  const char *ksrc = p.keys + token * p.key_stride_bytes + (int64_t)layer0 * p.n * Src::kBytes;
  const char *vsrc = p.values + token * p.value_stride_bytes + (int64_t)layer0 * p.n * Src::kBytes;
  const int cpr = p.chunks_per_row;
  const int total = 2 * nlayers * cpr;  // chunks this workgroup moves

  auto locate = [&](int c, int &r, int &col) {
    if constexpr (kPow2) {
      r = c >> p.chunk_shift;
      col = c & (cpr - 1);
    } else {
      r = (int)p.by_chunks.quotient((uint32_t)c);
      col = c - r * cpr;
    }
  };
  constexpr std::integral_constant<int, 0> kNone;
  constexpr std::integral_constant<int, kWholeAhead ? kUnroll : kUnroll / 2> kAhead;
  constexpr std::integral_constant<int, kUnroll> kAll;
  // independent 16-byte loads `from` ... `to` - 1 of a lane's kUnroll; lanes past the end load nothing
  auto load_part = [&](int c, uint4 (&v)[kUnroll], auto from, auto to) {
#pragma unroll
    for (int u = decltype(from)::value; u < decltype(to)::value; ++u) {
      const int cu = c + u * kBulkThreads;
      if (cu < total) {
        int r, col;
        locate(cu, r, col);
        const char *base = (r & 1) ? vsrc : ksrc;
        v[u] = load16_stream(base + ((int64_t)(r >> 1) * cpr + col) * 16);
      }
    }
  };

  // The first half of the first batch is requested together with the slot (source addresses do not depend on it), the
  // rest behind it: a padding token then throws half a batch away, or nothing in the shape of one chunk per lane.  With one
  // batch per workgroup and 30 % padding what the padding's whole first batches read was 22 % of a launch's traffic; with
  // nothing requested ahead CUs that hold a few short-lived workgroups wait for their slots.  Us per call in a graph, bf16 to
  // fp8, all / none / two of a lane's four chunks ahead: 8192 x 16 of 8 x 128 156.4 / 157.0 / 155.7 without padding, 145.8 /
  // 143.1 / 144.3 with 10 %, 124.9 / 110.9 / 117.3 with 30 %; without padding 512 x 40 23.7 / 24.2 / 23.8, 1024 x 16 18.7 /
  // 19.0 / 18.7, 512 x 16 10.2 / 10.0 / 9.9, 64 x 16 3.71 / 3.73 / 3.49; in the 1024-lane shape, all / none, 16384 x 40 762.7 /
  // 763.1 without padding, 695.9 / 687.3 with 10 %, 575 / 548 with 30 %.  Where the index list is scanned
  // the scan stands between the slot and the stores already, and batches are requested whole (half ahead, 448 x 16 of 3 x 96,
  // copied, 112 selected: 6.5 / 7.0).  By row map half ahead is level (2049 to 16384 tokens, 1476 calls of bf16 and fp32: the
  // middle one -0.2 %, with 30 % padding -0.4), fp32 sources gain as 16-bit ones do (with 30 % padding -2 %).
  // kWholeAhead: copies of 10 to 26 MB, which have no scale to wait for and whose workgroups all run side by side.  Their time
  // rises in steps (of 44 x 1 x 128 bf16 7 % at 18 MB and 28 % at 21), which come earlier with half of the batch ahead.  Us per call, whole / half: 512 x
  // 40 of 1 x 128 fp32 7.74 / 8.43, 843 x 44 of 1 x 128 bf16 7.13 / 7.78, 506 x 36 of 3 x 96 8.35 / 9.11, 289 x 36 of it 5.53 /
  // 5.75; of 391 drawn ones without padding half is 1.2 % slower in the mean and 10 % at the most, of 194 with 30 % padding 0.7 %
  // faster in the mean.
  const int64_t slot = p.slot_mapping[token];
  int64_t out_row = -1;
  if constexpr (kSelect == kSelectByRowMap) out_row = p.row_map[token];
  // by scan: every lane requests its share of the index list ahead of the source rows, like the slot, and compares
  // it with the token once the first batch is on its way; the output rows that name this token end up in `hits`
  constexpr int kIndicesPerLane = ARCTIC_SELECT_SCAN_MAX_INDICES / kBulkThreads;
  __shared__ int hits[kSelect == kSelectByScan ? ARCTIC_SELECT_SCAN_MAX_INDICES : 1];
  __shared__ int num_hits;
  [[maybe_unused]] int64_t mine[kIndicesPerLane];
  if constexpr (kSelect == kSelectByScan) {
#pragma unroll
    for (int k = 0; k < kIndicesPerLane; ++k) {
      const int j = threadIdx.x + k * kBulkThreads;
      mine[k] = -1;   // no token
      if (j < (int)p.num_out_rows)
        mine[k] = p.index_is_64 ? ((const int64_t *)p.indices)[j] : (int64_t)((const int32_t *)p.indices)[j];
    }
    if (threadIdx.x == 0) num_hits = 0;
  }
  // padding (or a slot outside the cache) writes no cache row; this and to_out below are uniform over the workgroup
  const bool to_cache = slot >= 0 && slot < p.num_slots;
  bool to_out = false;
  if constexpr (kSelect == kSelectByRowMap) to_out = out_row >= 0 && out_row < p.num_out_rows;
  int c = threadIdx.x;
  uint4 cur[kUnroll];
  if constexpr (kSelect == kSelectByScan) {
    load_part(c, cur, kNone, kAll);
  } else {
    load_part(c, cur, kNone, kAhead);
    __builtin_amdgcn_sched_barrier(0);   // ahead of the wait for the slot
    if (!to_cache && !to_out) return;
    load_part(c, cur, kAhead, kAll);
  }
  int nhits = 0;
  if constexpr (kSelect == kSelectByScan) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kIndicesPerLane; ++k)
      if (mine[k] == token) hits[atomicAdd(&num_hits, 1)] = threadIdx.x + k * kBulkThreads;
    __syncthreads();
    nhits = num_hits;
    to_out = nhits > 0;
    if (!to_cache && !to_out) return;   // uniform, and behind the scan's barriers
  }

  if (to_cache) {
    int64_t blk, off;
    if (slot < 0x7fffffffLL) {
      const uint32_t s32 = (uint32_t)slot;
      blk = p.by_block.quotient(s32);
      off = s32 - (uint32_t)blk * (uint32_t)p.block_size;
    } else {
      blk = slot / p.block_size;
      off = slot - blk * p.block_size;
    }
    const int64_t row_elem = blk * p.block_stride + off * (int64_t)p.n;

    // one lane per (layer, K|V) row of this token
    for (int r = threadIdx.x; r < 2 * nlayers; r += kBulkThreads) {
      const int layer = layer0 + (r >> 1);
      const bool is_v = r & 1;
      const void *base = is_v ? tab.value_cache[layer] : tab.key_cache[layer];
      RowDesc d;
      d.dst = (char *)base + row_elem * kDstElemBytes;
      d.inv = 0.0;
      if constexpr (!kCopy) {
        const float *sp = is_v ? tab.v_scale[layer] : tab.k_scale[layer];
        d.inv = 1.0 / (double)(*sp);
      }
      rows[r] = d;
    }
    __syncthreads();
  }
  char *kout = nullptr, *vout = nullptr;
  if constexpr (kSelect == kSelectByRowMap) {
    if (to_out) {
      kout = p.keys_out + out_row * p.out_key_stride_bytes + (int64_t)layer0 * p.n * Src::kBytes;
      vout = p.values_out + out_row * p.out_value_stride_bytes + (int64_t)layer0 * p.n * Src::kBytes;
    }
  }
  if constexpr (kSelect == kSelectByScan) {   // the columns of this workgroup's layers; the row is added per hit
    kout = p.keys_out + (int64_t)layer0 * p.n * Src::kBytes;
    vout = p.values_out + (int64_t)layer0 * p.n * Src::kBytes;
  }

  // Main loop: a batch is converted and stored, then the next one is requested.  (Requesting the next batch first,
  // so that it is in flight during the conversion, measures the same within half a per cent at every size and
  // placement: the other workgroups of the CU cover a workgroup's wait either way.)
  while (c < total) {
    const int cn = c + kUnroll * kBulkThreads;
    uint4 nxt[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int cu = c + u * kBulkThreads;
      if (cu < total) {
        int r, col;
        locate(cu, r, col);
        if (!kSelect || to_cache) emit_chunk<Src, Dst>(cur[u], rows[r], col);
        if constexpr (kSelect == kSelectByRowMap) {
          if (to_out) store16_stream(((r & 1) ? vout : kout) + ((int64_t)(r >> 1) * cpr + col) * 16, cur[u]);
        }
        if constexpr (kSelect == kSelectByScan) {
          const int64_t off = ((int64_t)(r >> 1) * cpr + col) * 16;
          for (int h = 0; h < nhits; ++h) {   // one hit unless the list names the token more than once
            const int64_t j = hits[h];
            store16_stream((r & 1) ? vout + j * p.out_value_stride_bytes + off : kout + j * p.out_key_stride_bytes + off,
                           cur[u]);
          }
        }
      }
    }
    load_part(cn, nxt, kNone, kAll);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) cur[u] = nxt[u];
    c = cn;
  }
}

template <typename Src, typename Dst, bool kPow2, int kBulkThreads, int kUnroll, int kSelect, int kLayers, bool kWholeAhead>
__global__ __launch_bounds__(kBulkThreads) void kv_write_bulk_kernel(const BulkParamsOf<kSelect> p,
                                                                         const LayerTables<kLayers> tab) {
  bulk_item<Src, Dst, kPow2, kBulkThreads, kUnroll, kSelect, kWholeAhead>(p, tab, blockIdx.x);
}

// Fallback for shapes or addresses that do not allow 16-byte accesses: one
// element per lane per step, any alignment.  Same arithmetic, no vector access.
template <typename SrcElem, typename Dst>
__global__ __launch_bounds__(kScalarThreads) void kv_write_bulk_scalar_kernel(
    const BulkSelectParams p, const LayerTables<kLayersPerLaunch> tab, const int src_dtype) {
  constexpr bool kCopy = std::is_same<Dst, Copy>::value;
  if (blockIdx.x < p.index_blocks) {  // the index list's own workgroups (select variant only)
    __shared__ int64_t todo_j[kScalarThreads], todo_t[kScalarThreads];
    __shared__ int count;
    const int n = p.select_mode == kSelectByScan
                      ? list_leftover_rows<kScalarThreads, kSelectByScan>(p, blockIdx.x, todo_j, todo_t, count)
                      : list_leftover_rows<kScalarThreads, kSelectByRowMap>(p, blockIdx.x, todo_j, todo_t, count);
    for (int e = 0; e < n; ++e) {
      const int64_t j = todo_j[e], t = todo_t[e];
      const SrcElem *ks = reinterpret_cast<const SrcElem *>(p.keys + t * p.key_stride_bytes);
      const SrcElem *vs = reinterpret_cast<const SrcElem *>(p.values + t * p.value_stride_bytes);
      SrcElem *ko = reinterpret_cast<SrcElem *>(p.keys_out + j * p.out_key_stride_bytes);
      SrcElem *vo = reinterpret_cast<SrcElem *>(p.values_out + j * p.out_value_stride_bytes);
      for (int64_t i = threadIdx.x; i < (int64_t)p.num_layers * p.n; i += kScalarThreads) {
        ko[i] = ks[i];
        vo[i] = vs[i];
      }
    }
    return;
  }
  const unsigned block = blockIdx.x - p.index_blocks;
  const int64_t token = block / (unsigned)p.groups_per_token;
  const int group = block - (unsigned)token * (unsigned)p.groups_per_token;
  const int layer0 = group * p.layers_per_group;
  const int nlayers = min(p.layers_per_group, p.num_layers - layer0);
  const int64_t slot = p.slot_mapping[token];
  // output rows of this token: the one the row map names, or all that a scan of the index list finds
  __shared__ int hits[ARCTIC_SELECT_SCAN_MAX_INDICES];
  __shared__ int num_hits;
  int nhits = 0;
  if (p.select_mode == kSelectByScan) {   // uniform
    if (threadIdx.x == 0) num_hits = 0;
    __syncthreads();
    for (int j = threadIdx.x; j < (int)p.num_out_rows; j += kScalarThreads) {
      const int64_t t = p.index_is_64 ? ((const int64_t *)p.indices)[j] : (int64_t)((const int32_t *)p.indices)[j];
      if (t == token) hits[atomicAdd(&num_hits, 1)] = j;
    }
    __syncthreads();
    nhits = num_hits;
  } else if (p.select_mode == kSelectByRowMap) {
    const int64_t out_row = p.row_map[token];
    if (out_row >= 0 && out_row < p.num_out_rows) {
      if (threadIdx.x == 0) hits[0] = (int)out_row;
      nhits = 1;
    }
    __syncthreads();
  }
  const bool to_cache = slot >= 0 && slot < p.num_slots;
  if (!to_cache && nhits == 0) return;
  const SrcElem *ks = reinterpret_cast<const SrcElem *>(p.keys + token * p.key_stride_bytes);
  const SrcElem *vs = reinterpret_cast<const SrcElem *>(p.values + token * p.value_stride_bytes);
  for (int h = 0; h < nhits; ++h) {
    const int64_t out_row = hits[h];
    SrcElem *ko = reinterpret_cast<SrcElem *>(p.keys_out + out_row * p.out_key_stride_bytes);
    SrcElem *vo = reinterpret_cast<SrcElem *>(p.values_out + out_row * p.out_value_stride_bytes);
    for (int64_t i = (int64_t)layer0 * p.n + threadIdx.x; i < (int64_t)(layer0 + nlayers) * p.n; i += kScalarThreads) {
      ko[i] = ks[i];
      vo[i] = vs[i];
    }
  }
  if (!to_cache) return;
  const int64_t blk = slot / p.block_size;
  const int64_t off = slot - blk * p.block_size;
  const int64_t row_elem = blk * p.block_stride + off * (int64_t)p.n;

  for (int l = layer0; l < layer0 + nlayers; ++l) {
    double kinv = 0.0, vinv = 0.0;
    if constexpr (!kCopy) {
      kinv = 1.0 / (double)(*tab.k_scale[l]);
      vinv = 1.0 / (double)(*tab.v_scale[l]);
    }
    for (int i = threadIdx.x; i < p.n; i += kScalarThreads) {
      const SrcElem k = ks[(int64_t)l * p.n + i];
      const SrcElem v = vs[(int64_t)l * p.n + i];
      if constexpr (kCopy) {
        ((SrcElem *)tab.key_cache[l])[row_elem + i] = k;
        ((SrcElem *)tab.value_cache[l])[row_elem + i] = v;
      } else {
        float kf, vf;
        if constexpr (sizeof(SrcElem) == 4) {
          kf = __uint_as_float((uint32_t)k);
          vf = __uint_as_float((uint32_t)v);
        } else if (src_dtype == ARCTIC_DTYPE_BF16) {
          kf = BF16::lo((uint32_t)k);
          vf = BF16::lo((uint32_t)v);
        } else {
          kf = F16::lo((uint32_t)k);
          vf = F16::lo((uint32_t)v);
        }
        const uint32_t wk = encode4<Dst>(div_by_scale(kf, kinv), 0.f, 0.f, 0.f);
        const uint32_t wv = encode4<Dst>(div_by_scale(vf, vinv), 0.f, 0.f, 0.f);
        ((uint8_t *)tab.key_cache[l])[row_elem + i] = (uint8_t)(wk & 0xffu);
        ((uint8_t *)tab.value_cache[l])[row_elem + i] = (uint8_t)(wv & 0xffu);
      }
    }
  }
}

// The per-layer pointers of a call, from the first layer of a launch on; scales are nullptr for a copy.
struct LayerPointers {
  const void *const *key_cache;
  const void *const *value_cache;
  const float *const *k_scale;
  const float *const *v_scale;
  template <int kLayers>
  void fill(LayerTables<kLayers> &tab, int count) const {   // the entries behind `count` are never read
    std::copy_n(key_cache, count, tab.key_cache);
    std::copy_n(value_cache, count, tab.value_cache);
    if (k_scale) std::copy_n(k_scale, count, tab.k_scale);
    if (v_scale) std::copy_n(v_scale, count, tab.v_scale);
  }
};

template <typename Src, typename Dst, int kSelect>
static void launch_vec_shape(const BulkSelectParams &p, const LayerPointers &layers, int64_t grid, bool wide,
                             bool whole_ahead, hipStream_t s) {
  const dim3 g((unsigned)grid);
#define ARCTIC_BULK_LAUNCH(POW2, LANES, UNROLL, LAYERS, WHOLE_AHEAD)                                                \
  do {                                                                                                             \
    LayerTables<LAYERS> tab;                                                                                       \
    layers.fill(tab, p.num_layers);                                                                                \
    launch<BulkParamsOf<kSelect>>(kv_write_bulk_kernel<Src, Dst, POW2, LANES, UNROLL, kSelect, LAYERS, WHOLE_AHEAD>, g, LANES, \
                                  s, p, tab);                                                                      \
  } while (0)
  if constexpr (kSelect == kSelectNone) {
    // The 256-lane shape is also that of the small launches, which cost what it takes to issue them: few layers leave
    // 1.5 KB of their arguments out.
    const bool few = p.num_layers <= kFewLayers;
#define ARCTIC_BULK_LAUNCH_256(WHOLE_AHEAD)                                                               \
  do {                                                                                                   \
    if (p.chunk_shift < 0 && few) ARCTIC_BULK_LAUNCH(false, 256, 4, kFewLayers, WHOLE_AHEAD);             \
    else if (p.chunk_shift < 0) ARCTIC_BULK_LAUNCH(false, 256, 4, kLayersPerLaunch, WHOLE_AHEAD);         \
    else if (few) ARCTIC_BULK_LAUNCH(true, 256, 4, kFewLayers, WHOLE_AHEAD);                              \
    else ARCTIC_BULK_LAUNCH(true, 256, 4, kLayersPerLaunch, WHOLE_AHEAD);                                 \
  } while (0)
    if (wide) {
      if (p.chunk_shift < 0) ARCTIC_BULK_LAUNCH(false, 1024, 1, kLayersPerLaunch, false);
      else ARCTIC_BULK_LAUNCH(true, 1024, 1, kLayersPerLaunch, false);   // 0.5-2 % faster than the same batch as 512 x 2
      return;
    }
    if constexpr (std::is_same<Dst, Copy>::value) {
      if (whole_ahead) {
        ARCTIC_BULK_LAUNCH_256(true);
        return;
      }
    }
    ARCTIC_BULK_LAUNCH_256(false);
#undef ARCTIC_BULK_LAUNCH_256
  } else {
    if (p.chunk_shift < 0) ARCTIC_BULK_LAUNCH(false, 256, 4, kLayersPerLaunch, false);
    else if (wide) ARCTIC_BULK_LAUNCH(true, 512, 2, kLayersPerLaunch, false);
    else ARCTIC_BULK_LAUNCH(true, 256, 4, kLayersPerLaunch, false);
  }
#undef ARCTIC_BULK_LAUNCH
}
template <typename Src, typename Dst>
static void launch_vec(const BulkSelectParams &p, const LayerPointers &layers, int64_t grid, bool wide,
                       bool whole_ahead, hipStream_t s) {
  switch (p.select_mode) {
    case kSelectByScan: launch_vec_shape<Src, Dst, kSelectByScan>(p, layers, grid, wide, whole_ahead, s); break;
    case kSelectByRowMap: launch_vec_shape<Src, Dst, kSelectByRowMap>(p, layers, grid, wide, whole_ahead, s); break;
    default: launch_vec_shape<Src, Dst, kSelectNone>(p, layers, grid, wide, whole_ahead, s); break;
  }
}
template <typename SrcElem, typename Dst>
static void launch_scalar(const BulkSelectParams &p, const LayerPointers &layers, int64_t grid, int src_dtype,
                          hipStream_t s) {
  LayerTables<kLayersPerLaunch> tab;
  layers.fill(tab, p.num_layers);
  hipLaunchKernelGGL((kv_write_bulk_scalar_kernel<SrcElem, Dst>), dim3((unsigned)grid),
                     dim3(kScalarThreads), 0, s, p, tab, src_dtype);
}

template <typename Dst>
static void dispatch_src(bool vec, bool wide, bool whole_ahead, int src_dtype, const BulkSelectParams &p,
                         const LayerPointers &layers, int64_t grid, hipStream_t s) {
  if (vec) {
    switch (src_dtype) {
      case ARCTIC_DTYPE_BF16: launch_vec<SrcBF16, Dst>(p, layers, grid, wide, whole_ahead, s); break;
      case ARCTIC_DTYPE_F16: launch_vec<SrcF16, Dst>(p, layers, grid, wide, whole_ahead, s); break;
      default: launch_vec<SrcF32, Dst>(p, layers, grid, wide, whole_ahead, s); break;
    }
  } else {
    if (src_dtype == ARCTIC_DTYPE_F32)
      launch_scalar<uint32_t, Dst>(p, layers, grid, src_dtype, s);
    else
      launch_scalar<uint16_t, Dst>(p, layers, grid, src_dtype, s);
  }
}

// row_map[t] = j where indices[j] == t, -1 where no j is: one workgroup, so that the fill is complete
// (barrier) before the rows are entered.  Tens of thousands of tokens at most: a few microseconds.
template <typename Index>
__global__ __launch_bounds__(1024) void build_row_map_kernel(int64_t *__restrict__ row_map, int64_t num_tokens,
                                                             const Index *__restrict__ indices, int64_t num_indices) {
  for (int64_t t = threadIdx.x; t < num_tokens; t += blockDim.x) row_map[t] = -1;
  __syncthreads();
  for (int64_t j = threadIdx.x; j < num_indices; j += blockDim.x) {
    const int64_t t = (int64_t)indices[j];
    if (t >= 0 && t < num_tokens) row_map[t] = j;
  }
}

static inline bool aligned(const void *p, uintptr_t a) { return ((uintptr_t)p % a) == 0; }

}  // namespace arctic

using namespace arctic;

// The rows a launch may also copy out (the select variant); row_map == nullptr: none.
struct SelectArgs {
  int mode;                  // kSelectNone / kSelectByRowMap / kSelectByScan
  const int64_t *row_map;    // kSelectByRowMap only
  void *keys_out;
  void *values_out;
  int64_t out_key_stride;    // elements
  int64_t out_value_stride;
  int64_t num_out_rows;
  const void *indices;       // the index list (num_out_rows entries); with a row map it may be nullptr
  int index_bytes;
  int64_t num_src_rows;      // rows of keys / values an index may name
};

static int bulk_entry(const char *fn, const void *keys, const void *values, int64_t key_stride, int64_t value_stride,
                      const void *const *key_cache_ptrs, const void *const *value_cache_ptrs,
                      const float *const *k_scale_ptrs, const float *const *v_scale_ptrs,
                      const int64_t *slot_mapping, int64_t num_tokens, int num_layers, int num_heads, int head_size,
                      int block_size, int64_t block_stride, int64_t num_blocks, int src_dtype, int kv_cache_dtype,
                      const SelectArgs &sel_in, void *stream, bool check_only = false) {
  if (num_layers == 0 || num_tokens == 0) return ARCTIC_OK;  // reference :87-89
  if (num_layers < 0 || num_layers > ARCTIC_MAX_LAYERS)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: num_layers=%d outside [0, %d]", fn, num_layers,
                ARCTIC_MAX_LAYERS);
  if (num_tokens < 0 || num_tokens > 0x7fffffffLL)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: num_tokens=%lld outside [0, 2^31)", fn, (long long)num_tokens);
  if (num_heads <= 0 || head_size <= 0 || block_size <= 0)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: num_heads, head_size and block_size must be positive", fn);
  if (num_blocks < 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: negative num_blocks", fn);
  if (src_dtype != ARCTIC_DTYPE_F32 && src_dtype != ARCTIC_DTYPE_F16 && src_dtype != ARCTIC_DTYPE_BF16)
    return fail(ARCTIC_ERR_UNSUPPORTED, "%s: Unsupported input type of kv cache: %d", fn, src_dtype);
  if (kv_cache_dtype != ARCTIC_KV_AUTO && kv_cache_dtype != ARCTIC_KV_FP8_E4M3 &&
      kv_cache_dtype != ARCTIC_KV_FP8_E5M2)
    return fail(ARCTIC_ERR_UNSUPPORTED, "%s: Unsupported data type of kv cache: %d", fn, kv_cache_dtype);
  if (!keys || !values || !slot_mapping || !key_cache_ptrs || !value_cache_ptrs)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null tensor pointer", fn);
  if (block_size > (1 << 20) || num_blocks > ((int64_t)1 << 40))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: block_size beyond 2^20 or num_blocks beyond 2^40", fn);
  {
    const int src_bytes = src_dtype == ARCTIC_DTYPE_F32 ? 4 : 2;
    const int64_t src_rows = sel_in.mode != kSelectNone && sel_in.indices ? std::max(num_tokens, sel_in.num_src_rows) : num_tokens;
    if (!pitch_ok(key_stride, src_rows, src_bytes) || !pitch_ok(value_stride, src_rows, src_bytes) ||
        !pitch_ok(block_stride, num_blocks, kv_cache_dtype == ARCTIC_KV_AUTO ? src_bytes : 1))
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: row or block pitch out of range", fn);
    if (sel_in.mode != kSelectNone && (!pitch_ok(sel_in.out_key_stride, sel_in.num_out_rows, src_bytes) ||
                                       !pitch_ok(sel_in.out_value_stride, sel_in.num_out_rows, src_bytes)))
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: negative number of output rows or row pitch out of range", fn);
  }
  SelectArgs sel = sel_in;
  if (sel.mode != kSelectNone) {
    if (sel.num_out_rows < 0 || sel.num_out_rows > 0x7fffffffLL || sel.out_key_stride < 0 || sel.out_value_stride < 0)
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: negative number of output rows or row pitch, or 2^31 output rows or more", fn);
    if (sel.num_out_rows == 0) sel.mode = kSelectNone;   // no row to copy to: the plain write
  }
  if (sel.mode != kSelectNone) {
    if (!sel.keys_out || !sel.values_out) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null keys_out or values_out", fn);
    if (sel.mode == kSelectByRowMap && !sel.row_map) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null row map", fn);
    if (sel.mode == kSelectByScan && (!sel.indices || sel.num_out_rows > ARCTIC_SELECT_SCAN_MAX_INDICES))
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: the index list is missing or longer than %d entries and there is no row map",
                  fn, ARCTIC_SELECT_SCAN_MAX_INDICES);
    if (sel.indices) {
      if (sel.index_bytes != 4 && sel.index_bytes != 8)
        return fail(ARCTIC_ERR_UNSUPPORTED, "%s: indices must be int32 or int64", fn);
      if (sel.num_src_rows < num_tokens)
        return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: keys / values have fewer rows (%lld) than slot_mapping (%lld)", fn,
                    (long long)sel.num_src_rows, (long long)num_tokens);
    }
  }
  const bool quant = kv_cache_dtype != ARCTIC_KV_AUTO;
  if (quant && (!k_scale_ptrs || !v_scale_ptrs))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: fp8 cache needs k_scales and v_scales", fn);
  const int64_t n64 = (int64_t)num_heads * head_size;
  if (n64 > (1 << 24)) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: num_heads*head_size too large", fn);
  const int n = (int)n64;
  for (int l = 0; l < num_layers; ++l) {
    if (!key_cache_ptrs[l] || !value_cache_ptrs[l])
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null cache pointer for layer %d", fn, l);
    if (quant && (!k_scale_ptrs[l] || !v_scale_ptrs[l]))
      return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null scale pointer for layer %d", fn, l);
  }

  const int es = src_dtype == ARCTIC_DTYPE_F32 ? 4 : 2;
  const int des = quant ? 1 : es;
  const int epc = 16 / es;  // elements per 16-byte chunk
  // 16-byte loads need aligned rows; stores are 16 B (copy), 8 B (fp8 from 16-bit) or 4 B (fp8 from fp32)
  const int store_bytes = quant ? epc : 16;
  // (a single source row needs no pitch; with an index list the index workgroups read rows up to num_src_rows)
  const bool one_source_row =
      (sel.mode != kSelectNone && sel.indices ? std::max(num_tokens, sel.num_src_rows) : num_tokens) == 1;
  bool vec = (n % epc == 0) && aligned(keys, 16) && aligned(values, 16) &&
             ((key_stride * es) % 16 == 0 || one_source_row) &&
             ((value_stride * es) % 16 == 0 || one_source_row) && ((block_stride * des) % store_bytes == 0);
  for (int l = 0; vec && l < num_layers; ++l)
    vec = aligned(key_cache_ptrs[l], store_bytes) && aligned(value_cache_ptrs[l], store_bytes);
  if (vec && sel.mode != kSelectNone)
    vec = aligned(sel.keys_out, 16) && aligned(sel.values_out, 16) &&
          ((sel.out_key_stride * es) % 16 == 0 || sel.num_out_rows <= 1) &&
          ((sel.out_value_stride * es) % 16 == 0 || sel.num_out_rows <= 1);

  hipStream_t s = (hipStream_t)stream;
  // More than kLayersPerLaunch layers take several launches.  Pass 0 plans every launch and checks its grid, so that
  // a call that is refused has launched nothing; pass 1 launches (a single launch is checked just before it is made).
  for (int pass = (check_only || num_layers > kLayersPerLaunch) ? 0 : 1; pass < (check_only ? 1 : 2); ++pass) {
    for (int first = 0; first < num_layers; first += kLayersPerLaunch) {
      const int count = std::min(kLayersPerLaunch, num_layers - first);
      const LayerPointers layers = {key_cache_ptrs + first, value_cache_ptrs + first, quant ? k_scale_ptrs + first : nullptr,
                                    quant ? v_scale_ptrs + first : nullptr};
      BulkSelectParams p;
      p.keys = (const char *)keys + (int64_t)first * n * es;
      p.values = (const char *)values + (int64_t)first * n * es;
      p.slot_mapping = slot_mapping;
      const bool select = sel.mode != kSelectNone;
      p.select_mode = sel.mode;
      p.row_map = sel.mode == kSelectByRowMap ? sel.row_map : nullptr;
      p.keys_out = select ? (char *)sel.keys_out + (int64_t)first * n * es : nullptr;
      p.values_out = select ? (char *)sel.values_out + (int64_t)first * n * es : nullptr;
      p.out_key_stride_bytes = sel.out_key_stride * es;
      p.out_value_stride_bytes = sel.out_value_stride * es;
      p.num_out_rows = select ? sel.num_out_rows : 0;
      p.indices = select ? sel.indices : nullptr;
      p.index_is_64 = sel.index_bytes == 8;
      p.num_tokens = num_tokens;
      p.num_src_rows = sel.num_src_rows;
      p.key_stride_bytes = key_stride * es;
      p.value_stride_bytes = value_stride * es;
      p.block_stride = block_stride;
      p.num_slots = num_blocks > 0 ? num_blocks * (int64_t)block_size : INT64_MAX;
      p.num_layers = count;
      p.n = n;
      p.block_size = block_size;
      p.chunks_per_row = vec ? n / epc : 0;
      p.chunk_shift = -1;
      if (vec && (p.chunks_per_row & (p.chunks_per_row - 1)) == 0) p.chunk_shift = __builtin_ctz(p.chunks_per_row);

      // A token's layers are split over `groups` workgroups.  Measured best on gfx950 (sweeps over the group count and
      // the shapes at 5 to 16384 tokens, 16, 33 and 40 layers, rows of 240 to 1024 elements):
      //  - as long as a batch (1024 chunks) per workgroup makes no more than about 2048 workgroups of 256 lanes, the eight
      //    per CU that run side by side, a workgroup has one batch, the layers that fit it whole: a second one, mostly a
      //    few chunks, costs a memory round trip and is what the last workgroups do (us in a graph, layers spread to at
      //    least one batch each / to at most one: 100 x 33 of 3 x 80 6.12 / 4.71, 500 x 33 of 3 x 96 9.7 / 9.1, 1000 x
      //    33 of 3 x 80 15.3 / 13.3).  Copies, which store twice as much, do so up to seven per
      //    CU: of 230 drawn ones with 1792 to 2048 workgroups, plain and selecting, the middle one is 4 % faster and the slowest
      //    are 5 to 6 % slower (316 x 31 of 10 x 64 11.5 / 12.1, 1002 x 14 of 6 x 96 12.5 / 13.0; selecting 993 x 7 of 16 x
      //    64 18.1 / 19.3), and so do plain fp8 rows of a power of two, whose second batch is a full layer or two (80 drawn, the
      //    middle one 3 % faster, 245 x 58 of 4 x 128 11.0 / 11.7, 493 x 14 of 8 x 128 10.8 / 11.3); other fp8 rows there
      //    gain 9 %, selecting ones of any length 11 %;
      //  - fewer than about 512 such workgroups leave CUs idle or with a wave or two per SIMD, whose instructions count
      //    then: more and smaller ones, a chunk per lane at the least (5 x 16 of 8 x 128 3.61 / 3.19, 5 x 40 of 3 x 96
      //    4.59 / 3.70, 30 x 16 of 8 x 128 3.80 / 3.49; from 800 workgroups on it is level, behind 2048 each one more
      //    costs: 512 x 40 of 3 x 96 in 4 groups 9.95, in 5 11.7).  Writes that select rows gain more, although each
      //    of their workgroups looks through the whole index list (fp8, all rows selected, in two to ten groups / in three to
      //    25: 1, 5, 20 and 64 x 16 of 8 x 128 4.42 / 3.25, 4.54 / 3.33, 4.72 / 3.70 and 5.23 / 4.45, 20 x 40 5.17 / 4.63, 20
      //    and 512 x 33 of 3 x 96 5.71 / 4.13 and 14.3 / 11.9; the row map serves lists too long for these launches);
      //  - more tokens, up to 8192: about two batches (8 layers of 8 x 128) per workgroup, never less than one each;
      //  - above that, the wide shape (batches of 1024 chunks by 1024 lanes, by 512 lanes when rows are selected as well)
      //    with up to five batches per workgroup (20 layers of 8 x 128 bf16) and at least about 1024 workgroups; a
      //    workgroup that would get less than two batches takes the 256-lane shape instead.
      // Rows that are no power of two long take the wide shape from 4097 tokens on where a workgroup has three batches or
      // more, however full the last one (us, 256 lanes / 1024, fp8: 5003 x 33 of 3 x 96 73.1 / 71.3, 16384 x 40 of 3 x 80
      // 295 / 276, 8193 x 61 of 5 x 80 346 / 306, three batches 70 % full 8193 x 36 of 3 x 80 129 / 122; of 300 drawn calls up
      // to 8192 tokens the middle one is 1 % faster and the slowest 2.7 % slower, of 540 above 3 % faster and 1.4 % slower).
      // With one or two batches a lane has too few loads in flight to pay for a CU that holds two workgroups only: 5437 x 12
      // of 5 x 64 28.4 / 33.8, 4097 x 32 of 3 x 64 31.9 / 36.3, 5101 x 40 of 3 x 64 49.3 / 52.3, 9066 x 4 of 1 x 832 23 %
      // slower; only copies, which store twice as much, gain there as well where a single batch comes out 7/8 and two 3/4
      // full (two at 75 %, 8000 x 32 of 3 x 64 75.8 / 73.3; one at 94 %, 6572 x 20 of it 39.3 / 38.5).
      int groups = 1;
      bool wide = false;
      if (vec) {
        constexpr int64_t kBatch = 1024, kSideBySide = 2048, kFewWorkgroups = 512, kFewestChunks = 256;
        const int64_t chunks_per_layer = 2LL * p.chunks_per_row;
        const auto ceil_div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
        const auto limit = [&](int64_t g) { return std::max<int64_t>(1, std::min<int64_t>(g, count)); };
        const int64_t min_layers = std::max<int64_t>(1, ceil_div(kBatch, chunks_per_layer));
        const bool ragged = p.chunk_shift < 0;
        const int64_t one_batch_groups = ceil_div(count, std::max<int64_t>(1, kBatch / chunks_per_layer));
        if (num_tokens > 8192 || (ragged && !select && num_tokens > 4096)) {
          const int64_t g = limit(std::max(ceil_div(1024, num_tokens), ceil_div(chunks_per_layer * count, 5 * kBatch)));
          const int64_t chunks = ceil_div(count, g) * chunks_per_layer, slots = ceil_div(chunks, kBatch) * kBatch;
          if (!ragged || select) wide = chunks >= 2 * kBatch;
          else wide = chunks > 2 * kBatch || (!quant && chunks * 8 >= slots * (slots == kBatch ? 7 : 6));
          if (wide) groups = (int)g;
        }
        if (wide) {
          // as above
        } else if (num_tokens > 8192) {
          groups = (int)limit(std::min(ceil_div(kSideBySide, num_tokens), count / min_layers));
        } else if (num_tokens * one_batch_groups <= (quant && (ragged || select) ? kSideBySide : kSideBySide * 7 / 8)) {
          const int64_t fewest_layers = std::max<int64_t>(1, ceil_div(kFewestChunks, chunks_per_layer));
          groups = (int)limit(std::max(one_batch_groups, std::min(kFewWorkgroups / num_tokens, ceil_div(count, fewest_layers))));
        } else {
          const int64_t want = std::max(ceil_div(count, std::max<int64_t>(1, ceil_div(2 * kBatch, chunks_per_layer))),
                                        ceil_div(kSideBySide, num_tokens));
          groups = (int)limit(std::min(want, count / min_layers));
        }
      } else {
        groups = (int)std::max<int64_t>(1, std::min<int64_t>(count, (2048 + num_tokens - 1) / num_tokens));
      }
      p.layers_per_group = (count + groups - 1) / groups;
      p.groups_per_token = (count + p.layers_per_group - 1) / p.layers_per_group;
      p.by_chunks = Divisor((uint32_t)std::max(1, p.chunks_per_row));
      p.by_block = Divisor((uint32_t)block_size);
      p.by_groups = Divisor((uint32_t)p.groups_per_token);
      // lanes of the shape launched below when rows are selected (the only case with index workgroups)
      const int lanes = !vec ? kScalarThreads : (wide && p.chunk_shift >= 0) ? 512 : 256;
      const int64_t index_blocks = p.indices ? (p.num_out_rows + lanes - 1) / lanes : 0;
      const int64_t grid = num_tokens * p.groups_per_token + index_blocks;
      p.index_blocks = (unsigned)index_blocks;
      if (grid > 0x7fffffffLL)
        return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: too many tokens (%lld)", fn, (long long)num_tokens);
      if (pass == 0) continue;
      // Copies of 10 to 26 MB request their whole first batch ahead of the slot (bulk_item has why).  Below, half ahead is level
      // (padding 0 and 30 %: 8 to 9 MB -0.3 and -2 %), and so it is above (26 to 28 MB +0.4 and -3, 34 to 40 MB 0 and -4).
      const double source_mb = 2e-6 * num_tokens * count * n * es;
      const bool whole_ahead = !quant && !select && source_mb >= 10 && source_mb < 26;

      switch (kv_cache_dtype) {
        case ARCTIC_KV_AUTO: dispatch_src<Copy>(vec, wide, whole_ahead, src_dtype, p, layers, grid, s); break;
        case ARCTIC_KV_FP8_E4M3: dispatch_src<E4M3>(vec, wide, whole_ahead, src_dtype, p, layers, grid, s); break;
        default: dispatch_src<E5M2>(vec, wide, whole_ahead, src_dtype, p, layers, grid, s); break;
      }
      const int rc = check_launch(fn);
      if (rc) return rc;
    }
  }
  return ARCTIC_OK;
}

extern "C" int arctic_reshape_and_cache_flash_bulk(
    const void *keys, const void *values, int64_t key_stride, int64_t value_stride,
    const void *const *key_cache_ptrs, const void *const *value_cache_ptrs,
    const float *const *k_scale_ptrs, const float *const *v_scale_ptrs,
    const int64_t *slot_mapping, int64_t num_tokens, int num_layers, int num_heads,
    int head_size, int block_size, int64_t block_stride, int64_t num_blocks, int src_dtype,
    int kv_cache_dtype, void *stream) {
  const SelectArgs none = {kSelectNone, nullptr, nullptr, nullptr, 0, 0, 0, nullptr, 0, 0};
  return bulk_entry("reshape_and_cache_flash_bulk", keys, values, key_stride, value_stride, key_cache_ptrs,
                    value_cache_ptrs, k_scale_ptrs, v_scale_ptrs, slot_mapping, num_tokens, num_layers, num_heads,
                    head_size, block_size, block_stride, num_blocks, src_dtype, kv_cache_dtype, none, stream);
}

extern "C" int arctic_reshape_and_cache_flash_bulk_select(
    const void *keys, const void *values, int64_t key_stride, int64_t value_stride,
    const void *const *key_cache_ptrs, const void *const *value_cache_ptrs,
    const float *const *k_scale_ptrs, const float *const *v_scale_ptrs,
    const int64_t *slot_mapping, int64_t num_tokens, int num_layers, int num_heads,
    int head_size, int block_size, int64_t block_stride, int64_t num_blocks, int src_dtype,
    int kv_cache_dtype, const int64_t *row_map, const void *indices, int index_bytes, int64_t num_indices,
    int64_t num_src_rows, void *keys_out, void *values_out, int64_t out_key_stride, int64_t out_value_stride,
    void *stream) {
  const char *fn = "reshape_and_cache_flash_bulk_select";
  // a row map is used when one is given; without one the token workgroups scan the index list themselves
  const SelectArgs sel = {row_map ? kSelectByRowMap : kSelectByScan, row_map, keys_out, values_out, out_key_stride,
                          out_value_stride, num_indices, indices, index_bytes, num_src_rows};
  return bulk_entry(fn, keys, values, key_stride, value_stride, key_cache_ptrs, value_cache_ptrs, k_scale_ptrs,
                    v_scale_ptrs, slot_mapping, num_tokens, num_layers, num_heads, head_size, block_size, block_stride,
                    num_blocks, src_dtype, kv_cache_dtype, sel, stream);
}

static int build_row_map(const char *fn, int64_t *row_map, int64_t num_tokens, const void *indices, int index_bytes,
                         int64_t num_indices, void *stream) {
  if (index_bytes != 4 && index_bytes != 8) return fail(ARCTIC_ERR_UNSUPPORTED, "%s: indices must be int32 or int64", fn);
  if (num_tokens < 0 || num_indices < 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: negative size", fn);
  if (num_tokens == 0) return ARCTIC_OK;
  if (!row_map || (num_indices > 0 && !indices)) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null pointer", fn);
  hipStream_t s = (hipStream_t)stream;
  if (index_bytes == 8)
    hipLaunchKernelGGL(build_row_map_kernel<int64_t>, dim3(1), dim3(1024), 0, s, row_map, num_tokens,
                       (const int64_t *)indices, num_indices);
  else
    hipLaunchKernelGGL(build_row_map_kernel<int32_t>, dim3(1), dim3(1024), 0, s, row_map, num_tokens,
                       (const int32_t *)indices, num_indices);
  return check_launch(fn);
}

extern "C" int arctic_build_row_map(int64_t *row_map, int64_t num_tokens, const void *indices, int index_bytes,
                                    int64_t num_indices, void *stream) {
  return build_row_map("build_row_map", row_map, num_tokens, indices, index_bytes, num_indices, stream);
}

// ---- the select variant that allocates nothing ---------------------------------------------------------------
// The row map of arctic_reshape_and_cache_flash_bulk_select_static lives in this array instead of a workspace
// the caller brings in: 8 bytes per token, 2 MiB, held by every GPU the library has run on until the process
// ends.  In host code `scratch` is only a handle for the symbol; the array's address on a device comes from
// hipGetSymbolAddress with that device current, is looked up once per device and is what the kernels receive.
static __device__ __align__(256) int64_t scratch[ARCTIC_SELECT_STATIC_MAX_TOKENS];

namespace {
constexpr int kMaxDevices = 64;
// Per device: its copy of `scratch` (nullptr until first asked for), and what orders the calls that use it.  The
// array is shared by every call on the GPU, so a call on another stream than the last one first makes its stream
// wait for `last_use`, an event recorded behind the last call's kernels: calls on different streams then use the
// array one after the other instead of racing on it.  Under stream capture nothing of this is recorded.
struct DeviceScratch {
  int64_t *ptr = nullptr;
  hipEvent_t last_use = nullptr;
  hipStream_t last_stream = nullptr;
  bool used = false;
};
std::mutex g_scratch_mutex;
DeviceScratch g_scratch[kMaxDevices];
}  // namespace

static int scratch_on_current_device(const char *fn, DeviceScratch **out) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return fail(ARCTIC_ERR_LAUNCH, "%s: hipGetDevice failed: %s", fn, hipGetErrorString(err));
  if (dev < 0 || dev >= kMaxDevices) return fail(ARCTIC_ERR_UNSUPPORTED, "%s: device index %d not supported", fn, dev);
  DeviceScratch &d = g_scratch[dev];
  if (!d.ptr) {
    void *ptr = nullptr;
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !ptr)
      return fail(ARCTIC_ERR_LAUNCH, "%s: hipGetSymbolAddress failed on device %d: %s", fn, dev, hipGetErrorString(err));
    err = hipEventCreateWithFlags(&d.last_use, hipEventDisableTiming);
    if (err != hipSuccess)
      return fail(ARCTIC_ERR_LAUNCH, "%s: hipEventCreateWithFlags failed on device %d: %s", fn, dev, hipGetErrorString(err));
    d.ptr = (int64_t *)ptr;
  }
  *out = &d;
  return ARCTIC_OK;
}

extern "C" int arctic_reshape_and_cache_flash_bulk_select_static(
    const void *keys, const void *values, int64_t key_stride, int64_t value_stride,
    const void *const *key_cache_ptrs, const void *const *value_cache_ptrs,
    const float *const *k_scale_ptrs, const float *const *v_scale_ptrs,
    const int64_t *slot_mapping, int64_t num_tokens, int num_layers, int num_heads,
    int head_size, int block_size, int64_t block_stride, int64_t num_blocks, int src_dtype,
    int kv_cache_dtype, const void *indices, int index_bytes, int64_t num_indices, int64_t num_src_rows,
    void *keys_out, void *values_out, int64_t out_key_stride, int64_t out_value_stride, void *stream) {
  const char *fn = "reshape_and_cache_flash_bulk_select_static";
  if (num_tokens > ARCTIC_SELECT_STATIC_MAX_TOKENS)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT,
                "%s: num_tokens=%lld exceeds the %d tokens the static row map holds; use "
                "arctic_reshape_and_cache_flash_bulk_select with a row map of the caller's",
                fn, (long long)num_tokens, ARCTIC_SELECT_STATIC_MAX_TOKENS);
  if (num_indices < 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: negative number of indices", fn);
  if (num_indices > 0 && !indices) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null indices", fn);
  // short index lists are scanned by the token workgroups and need no row map; longer ones get theirs in `scratch`
  if (num_layers == 0 || num_tokens <= 0 || num_indices <= ARCTIC_SELECT_SCAN_MAX_INDICES) {
    const SelectArgs sel = {kSelectByScan, nullptr, keys_out, values_out, out_key_stride, out_value_stride, num_indices,
                            indices, index_bytes, num_src_rows};
    return bulk_entry(fn, keys, values, key_stride, value_stride, key_cache_ptrs, value_cache_ptrs, k_scale_ptrs,
                      v_scale_ptrs, slot_mapping, num_tokens, num_layers, num_heads, head_size, block_size,
                      block_stride, num_blocks, src_dtype, kv_cache_dtype, sel, stream);
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);   // one call at a time plans its use of the array
  DeviceScratch *d = nullptr;
  int rc = scratch_on_current_device(fn, &d);
  if (rc) return rc;
  const SelectArgs sel = {kSelectByRowMap, d->ptr, keys_out, values_out, out_key_stride, out_value_stride, num_indices,
                          indices, index_bytes, num_src_rows};
  // every argument is checked before the first kernel is enqueued: a call that is refused has launched nothing
  rc = bulk_entry(fn, keys, values, key_stride, value_stride, key_cache_ptrs, value_cache_ptrs, k_scale_ptrs,
                  v_scale_ptrs, slot_mapping, num_tokens, num_layers, num_heads, head_size, block_size, block_stride,
                  num_blocks, src_dtype, kv_cache_dtype, sel, stream, /*check_only=*/true);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess) capture = hipStreamCaptureStatusNone;
  const bool eager = capture == hipStreamCaptureStatusNone;
  if (eager && d->used && d->last_stream != s) {
    const hipError_t err = hipStreamWaitEvent(s, d->last_use, 0);
    if (err != hipSuccess) return fail(ARCTIC_ERR_LAUNCH, "%s: hipStreamWaitEvent failed: %s", fn, hipGetErrorString(err));
  }
  // every entry below num_tokens is rewritten, so nothing of an earlier call is seen
  rc = build_row_map(fn, d->ptr, num_tokens, indices, index_bytes, num_indices, stream);
  if (rc) return rc;
  rc = bulk_entry(fn, keys, values, key_stride, value_stride, key_cache_ptrs, value_cache_ptrs, k_scale_ptrs,
                  v_scale_ptrs, slot_mapping, num_tokens, num_layers, num_heads, head_size, block_size, block_stride,
                  num_blocks, src_dtype, kv_cache_dtype, sel, stream);
  if (eager) {
    const hipError_t err = hipEventRecord(d->last_use, s);
    if (err != hipSuccess && rc == ARCTIC_OK)
      rc = fail(ARCTIC_ERR_LAUNCH, "%s: hipEventRecord failed: %s", fn, hipGetErrorString(err));
    d->last_stream = s;
    d->used = true;
  }
  return rc;
}
