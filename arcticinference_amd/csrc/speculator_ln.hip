// Speculator "LayerNorm" (RMS norm with optional scale and shift) for gfx950.
//
// Replaces speculator_ln_cuda and its kernels
// (csrc/custom_ops/speculator_ln.cu:21-252 in the reference).
//
// One workgroup per row.  On the vector path every lane keeps its 16-byte
// chunks of the row in registers between the sum of squares and the scaling, so
// the row is read from HBM once (the reference reads it twice); the sum is a DPP
// wave reduction followed by a small LDS combine.  Rows that are only element-aligned
// take the same kernel with accesses at any alignment.
//
// The same kernel also carries the element-wise steps the speculator runs around
// this norm (arctic_speculator.py:296-307,733-734,809-816), each with the rounding
// of the separate PyTorch op it stands for:
//   x   = round(in + alpha * z)        states.add_(z, alpha=...)      (optional)
//   y   = round(x * inv_rms * w + b)   speculator_ln
//   y   = round(gelu(y))               nn.GELU()                      (optional)
//   out = round(y * out_scale)         ln0(x) / sqrt(2)               (optional)
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "activations.hpp"
#include "common.hpp"

namespace arctic {

// A launch's arguments, in one piece (common.hpp says what that is worth).
struct LnParams {
  char *out;
  const char *in;
  const char *weight;       // may be nullptr, like bias
  const char *bias;
  const char *z;            // nullptr: no add
  const int64_t *z_index;   // row of z to add to each row (an embedding lookup); nullptr = the row itself
  int64_t in_row_stride_bytes;
  int64_t z_row_stride_bytes;
  int64_t z_rows;           // rows of z when z_index is given; an index is clamped into [0, z_rows)
  int hidden;
  int waves;                // of the workgroup
  float inv_hidden;         // 1 / hidden
  float eps;
  float alpha;
  float out_scale;          // applied when != 1
  int activation;           // ARCTIC_ACT_* (the vector kernels take it as a template argument)
};

template <typename T>
__device__ __forceinline__ float glue_tail(float y, const LnParams &g, int activation) {
  if (activation != ARCTIC_ACT_NONE) {
    y = T::requant(y);
    y = activation == ARCTIC_ACT_GELU ? gelu_erf(y) : gelu_tanh(y);
  }
  if (g.out_scale != 1.0f) y = T::requant(y) * g.out_scale;
  return y;
}

// kAnyRow: rows that are only element-aligned (odd widths, pitches or bases): accesses at any alignment, and the last chunk
// of a width that is no multiple of 8 overlaps the one before it (common.hpp).  Bound like the aligned rows by the node's
// start and two dependent round trips; element by element and in two passes over the row (as such rows went before) every
// pass was a round trip per 256 elements.
// kGlue: what surrounds the norm: nothing (kPlain), or an add and a scale with or without the activation of that code - a
// launch of few rows waits for its instructions as well, and a kernel that holds both activations is twice as long (us per
// call in a graph, chosen at run time / here: embedding + add + norm + GELU of 64 x 2880 3.09 / 2.90, 1 x 4096 2.78 / 2.56,
// the scaled norm of 7 x 4096 2.20 / 2.10).
constexpr int kPlain = -1;
template <typename T, int kChunksPerThread, int kGlue, bool kAnyRow>
__global__ __launch_bounds__(1024) void spec_ln_vec_kernel(const LnParams p) {
  __shared__ float slots[16];
  const char *__restrict__ weight = p.weight, *__restrict__ bias = p.bias;
  const int hidden = p.hidden, lanes = p.waves * 64;
  const int chunks = kAnyRow ? (hidden + 7) >> 3 : hidden >> 3;
  auto offset = [&](int c) { return kAnyRow ? (int64_t)Place(c, hidden).off : (int64_t)c * 16; };
  const char *__restrict__ row_in = p.in + (int64_t)blockIdx.x * p.in_row_stride_bytes;
  char *__restrict__ row_out = p.out + (int64_t)blockIdx.x * hidden * 2;

  uint4 raw[kChunksPerThread], wv[kChunksPerThread], bv[kChunksPerThread];
  float ss = 0.f;
  // scale / shift first: they are cache resident and memory returns loads in issue
  // order, so asking for them after the row sum would add a full round trip
#pragma unroll
  for (int k = 0; k < kChunksPerThread; ++k) {
    const int c = threadIdx.x + k * lanes;
    if (weight && c < chunks) wv[k] = load16<kAnyRow>(weight + offset(c));
    if (bias && c < chunks) bv[k] = load16<kAnyRow>(bias + offset(c));
  }
#pragma unroll
  for (int k = 0; k < kChunksPerThread; ++k) {
    const int c = threadIdx.x + k * lanes;
    raw[k] = make_uint4(0, 0, 0, 0);
    if (c < chunks) raw[k] = load16_stream<kAnyRow>(row_in + offset(c));
  }
  if (kGlue != kPlain && p.z) {
    int64_t z_at = blockIdx.x;
    if (p.z_index) z_at = min(max(p.z_index[blockIdx.x], (int64_t)0), p.z_rows - 1);
    const char *row_z = p.z + z_at * p.z_row_stride_bytes;
    uint4 zr[kChunksPerThread];
#pragma unroll
    for (int k = 0; k < kChunksPerThread; ++k) {
      const int c = threadIdx.x + k * lanes;
      zr[k] = make_uint4(0, 0, 0, 0);
      if (c < chunks) zr[k] = load16_stream<kAnyRow>(row_z + offset(c));
    }
#pragma unroll
    for (int k = 0; k < kChunksPerThread; ++k) {
      float x[8], z[8];
      unpack8<T>(raw[k], x);
      unpack8<T>(zr[k], z);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = fmaf(p.alpha, z[j], x[j]);
      raw[k] = pack8<T>(x);   // the sum stands in the tensor's own type, as after the in-place add
    }
  }
#pragma unroll
  for (int k = 0; k < kChunksPerThread; ++k) {
    float x[8];
    unpack8<T>(raw[k], x);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (!kAnyRow || j >= Place(threadIdx.x + k * lanes, hidden).repeated) ss += x[j] * x[j];
  }
  const float total = block_sum(ss, slots, p.waves);
  const float inv = rsqrtf(total * p.inv_hidden + p.eps);

#pragma unroll
  for (int k = 0; k < kChunksPerThread; ++k) {
    const int c = threadIdx.x + k * lanes;
    if (c >= chunks) continue;
    float x[8];
    unpack8<T>(raw[k], x);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] *= inv;
    if (weight) {
      float w[8];
      unpack8<T>(wv[k], w);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= w[j];
    }
    if (bias) {
      float b[8];
      unpack8<T>(bv[k], b);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] += b[j];
    }
    if (kGlue != kPlain) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = glue_tail<T>(x[j], p, kGlue);
    }
    store16_stream<kAnyRow>(row_out + offset(c), pack8<T>(x));
  }
}

// What is left (short unaligned rows, rows beyond 65536 elements): element-wise, two passes over the row.
constexpr int kScalarLanes = 256;
template <typename T>
__global__ __launch_bounds__(kScalarLanes) void spec_ln_scalar_kernel(const LnParams p) {
  __shared__ float slots[16];
  const uint16_t *__restrict__ weight = (const uint16_t *)p.weight, *__restrict__ bias = (const uint16_t *)p.bias;
  const int hidden = p.hidden;
  const uint16_t *__restrict__ row_in = (const uint16_t *)(p.in + (int64_t)blockIdx.x * p.in_row_stride_bytes);
  int64_t z_at = blockIdx.x;
  if (p.z && p.z_index) z_at = min(max(p.z_index[blockIdx.x], (int64_t)0), p.z_rows - 1);
  const uint16_t *row_z = p.z ? (const uint16_t *)(p.z + z_at * p.z_row_stride_bytes) : nullptr;
  uint16_t *__restrict__ row_out = (uint16_t *)p.out + (int64_t)blockIdx.x * hidden;
  auto element = [&](int j) {
    float x = T::lo(row_in[j]);
    if (row_z) x = T::requant(fmaf(p.alpha, T::lo(row_z[j]), x));
    return x;
  };
  float ss = 0.f;
  for (int j = threadIdx.x; j < hidden; j += kScalarLanes) {
    const float x = element(j);
    ss += x * x;
  }
  const float total = block_sum(ss, slots, kScalarLanes / 64);
  const float inv = rsqrtf(total * p.inv_hidden + p.eps);
  for (int j = threadIdx.x; j < hidden; j += kScalarLanes) {
    float y = element(j) * inv;
    if (weight) y *= T::lo(weight[j]);
    if (bias) y += T::lo(bias[j]);
    row_out[j] = (uint16_t)T::round_bits(glue_tail<T>(y, p, p.activation));
  }
}

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

template <typename T>
static void launch_ln(LnParams p, int64_t rows, hipStream_t s) {
  const int activation = p.activation, hidden = p.hidden, chunks = (hidden + 7) / 8;
  const bool aligned = (hidden % 8 == 0) && (p.in_row_stride_bytes % 16 == 0 || rows == 1) && aligned16(p.in) &&
                       aligned16(p.out) && aligned16(p.weight) && aligned16(p.bias) &&   /* null counts as aligned */
                       (!p.z || (aligned16(p.z) && (p.z_row_stride_bytes % 16 == 0 || (rows == 1 && !p.z_index))));
  const bool plain = !p.z && activation == ARCTIC_ACT_NONE && p.out_scale == 1.0f;
  const dim3 grid((unsigned)rows);
  // Rows that are not 16-byte aligned take the same kernel with accesses at any alignment.  Us per call in a graph, element
  // by element / in chunks: 300 x 1537 fp16 5.5 / 3.3, 64 x 4096 pitched by 4099 7.0 / 2.7, 4000 x 4097 34.6 / 17.5 (3.7
  // TB/s), 300 x 20000 pitched by 20001 57 / 9.9, 300 x 65535 171 / 34 (eight chunks per lane, some of them in scratch);
  // 4000 x 160 4.7 / 3.6 and 300 x 100 level at 2.2, so that rows of fewer than 128 elements, where a single wave would do
  // a row's work, stay with the element-wise kernel.
  constexpr int kShortRow = 128;
  if (hidden >= (aligned ? 8 : kShortRow) && chunks <= 8 * 1024) {
    int cpt = 1;
    while (cpt < 8 && (chunks + cpt - 1) / cpt > 1024) cpt *= 2;
    int threads = (chunks + cpt - 1) / cpt;
    threads = std::max(64, (threads + 63) & ~63);
    p.waves = threads / 64;
#define ARCTIC_LN_LAUNCH_AS(CPT, GLUE, ANY) \
  launch(spec_ln_vec_kernel<T, CPT, GLUE, ANY>, grid, threads, s, p)
#define ARCTIC_LN_LAUNCH_GLUE(CPT, GLUE)                    \
  do {                                                      \
    if (aligned) ARCTIC_LN_LAUNCH_AS(CPT, GLUE, false);     \
    else ARCTIC_LN_LAUNCH_AS(CPT, GLUE, true);              \
  } while (0)
#define ARCTIC_LN_LAUNCH(CPT)                                                                          \
  do {                                                                                                 \
    if (plain) ARCTIC_LN_LAUNCH_GLUE(CPT, kPlain);                                                     \
    else if (activation == ARCTIC_ACT_NONE) ARCTIC_LN_LAUNCH_GLUE(CPT, ARCTIC_ACT_NONE);          \
    else if (activation == ARCTIC_ACT_GELU) ARCTIC_LN_LAUNCH_GLUE(CPT, ARCTIC_ACT_GELU);          \
    else ARCTIC_LN_LAUNCH_GLUE(CPT, ARCTIC_ACT_GELU_TANH);                                             \
  } while (0)
    switch (cpt) {
      case 1: ARCTIC_LN_LAUNCH(1); break;
      case 2: ARCTIC_LN_LAUNCH(2); break;
      case 4: ARCTIC_LN_LAUNCH(4); break;
      default: ARCTIC_LN_LAUNCH(8); break;
    }
#undef ARCTIC_LN_LAUNCH
#undef ARCTIC_LN_LAUNCH_GLUE
#undef ARCTIC_LN_LAUNCH_AS
  } else {
    launch(spec_ln_scalar_kernel<T>, grid, kScalarLanes, s, p);
  }
}

}  // namespace arctic

using namespace arctic;

// What surrounds the norm, as in LnParams.
struct LnGlue {
  const char *z;
  int64_t z_row_stride_bytes;
  const int64_t *z_index;
  int64_t z_rows;
  float alpha;
  int activation;
  float out_scale;
};

static int ln_entry(const char *fn, void *out, const void *in, const void *weight, const void *bias,
                    int64_t rows, int hidden, int64_t in_row_stride, float eps, const LnGlue &glue, int dtype,
                    void *stream) {
  if (dtype != ARCTIC_DTYPE_F16 && dtype != ARCTIC_DTYPE_BF16)
    return fail(ARCTIC_ERR_UNSUPPORTED, "%s: only fp16 and bf16 are supported.", fn);
  if (hidden <= 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: hidden size must be > 0", fn);
  if (hidden > (1 << 30)) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: hidden size beyond 2^30", fn);
  if (rows < 0 || rows > 0x7fffffffLL) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: bad row count", fn);
  if (glue.activation != ARCTIC_ACT_NONE && glue.activation != ARCTIC_ACT_GELU &&
      glue.activation != ARCTIC_ACT_GELU_TANH)
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: unknown activation %d", fn, glue.activation);
  if (rows == 0) return ARCTIC_OK;
  if (!out || !in) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null tensor pointer", fn);
  if (!pitch_ok(in_row_stride, rows, 2) || !pitch_ok(hidden, rows, 2))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: row pitch out of range", fn);
  const LnParams p = {(char *)out, (const char *)in, (const char *)weight, (const char *)bias, glue.z, glue.z_index,
                      in_row_stride * 2, glue.z_row_stride_bytes, glue.z_rows, hidden, 0, 1.0f / (float)hidden, eps,
                      glue.alpha, glue.out_scale, glue.activation};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ARCTIC_DTYPE_BF16) launch_ln<BF16>(p, rows, s);
  else launch_ln<F16>(p, rows, s);
  return check_launch(fn);
}

extern "C" int arctic_speculator_ln(void *out, const void *in, const void *weight, const void *bias,
                                    int64_t rows, int hidden, int64_t in_row_stride, float eps, int dtype,
                                    void *stream) {
  const LnGlue none = {nullptr, 0, nullptr, 0, 0.0f, ARCTIC_ACT_NONE, 1.0f};
  return ln_entry("speculator_ln", out, in, weight, bias, rows, hidden, in_row_stride, eps, none, dtype, stream);
}

extern "C" int arctic_speculator_add_ln_act(void *out, const void *in, const void *z, const void *weight,
                                            const void *bias, int64_t rows, int hidden, int64_t in_row_stride,
                                            int64_t z_row_stride, float alpha, float eps, int activation,
                                            float out_scale, int dtype, void *stream) {
  if (!pitch_ok(z_row_stride, rows, 2))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "speculator_add_ln_act: row pitch of z out of range");
  const LnGlue glue = {(const char *)z, z_row_stride * 2, nullptr, 0, alpha, activation, out_scale};
  return ln_entry("speculator_add_ln_act", out, in, weight, bias, rows, hidden, in_row_stride, eps, glue, dtype,
                  stream);
}

extern "C" int arctic_speculator_embed_add_ln_act(void *out, const void *in, const void *emb_table,
                                                  const int64_t *token_ids, const void *weight, const void *bias,
                                                  int64_t rows, int hidden, int64_t in_row_stride, int64_t emb_row_stride,
                                                  int64_t num_embeddings, float alpha, float eps, int activation,
                                                  float out_scale, int dtype, void *stream) {
  const char *fn = "speculator_embed_add_ln_act";
  if (rows > 0 && (!emb_table || !token_ids)) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: null embedding table or token ids", fn);
  if (rows > 0 && num_embeddings <= 0) return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: the embedding table has no rows", fn);
  if (!pitch_ok(emb_row_stride, num_embeddings, 2))
    return fail(ARCTIC_ERR_INVALID_ARGUMENT, "%s: row pitch of the embedding table out of range", fn);
  const LnGlue glue = {(const char *)emb_table, emb_row_stride * 2, token_ids, num_embeddings, alpha, activation, out_scale};
  return ln_entry(fn, out, in, weight, bias, rows, hidden, in_row_stride, eps, glue, dtype, stream);
}
