// Kernels that bench.py times next to the library's: what the same bytes cost on this GPU when nothing is
// computed, and what the reference's own launch decompositions of two operators cost on it.  Measurement aid only;
// nothing in the package uses it.
//
//   floor_lstm_traffic   the loads and stores of sum_lstm (nine 16-byte loads per lane from the rows of
//                        states, z4 and prev_cell, two 16-byte stores), one workgroup per row, no arithmetic
//   floor_lstm_traffic_staged  the same traffic requested in the stages of the library's staged kernel, each stage
//                        waiting for what its arithmetic would read, no arithmetic
//   floor_ln_traffic     the load and the store of speculator_ln (one 16-byte chunk per lane, one workgroup per row)
//   floor_row_read       the loads of the row-argmax kernel (one workgroup per row), nothing computed
//   floor_node           an empty kernel, or one that makes a single memory round trip: the fixed cost of a node
//   floor_valu_rate      chains of one vector-ALU operation, for its issue rate per SIMD
//   floor_stream         load-only, store-only or a 2:1 load:store stream in 64 KiB pieces, the pieces dealt
//                        round robin over up to three buffers (which the caller places in different regions
//                        of the HBM); the 2:1 stream also with its stores scattered as rows of 1 KiB
//   floor_write_per_layer_and_token  the bf16 -> e4m3 bulk write in the launch decomposition of the reference's kernel
//                        (csrc/custom_ops/reshape_and_cache_flash_bulk.cu:12-60, 133-135), written for this GPU: what
//                        that decomposition costs here, next to the library's
//   floor_sum_lstm_three_passes  sum_lstm (bf16, exact GELU) in the decomposition of the reference's kernel
//                        (csrc/custom_ops/sum_lstm.cu:28-191, launched :401-418): 128 lanes per row, three passes over
//                        global memory, two block sums, the C library's expf and erff
//   floor_ln_two_passes  speculator_ln (bf16, weight and bias) in the reference's decomposition
//                        (csrc/custom_ops/speculator_ln.cu:21-107, launched :203-207): 256 lanes per row, the row read
//                        twice from global memory with a block sum between
//   floor_stream_resident the scattered 2:1 stream once more, shaped for bandwidth alone: as many workgroups of 1024
//                        lanes as stay resident (one or two per CU), each looping over pieces with all of a piece's
//                        loads (4 or 8 per lane) requested before the first store
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cstdint>

#include "arcticinference_amd/csrc/common.hpp"   // 16-byte chunks of bf16 and their conversion to and from fp32

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__global__ void lstm_traffic_kernel(const char *s, const char *z, const char *pc, char *out_state, char *out_cell,
                                    int D) {
  const int chunks = D / 8;
  const int c = threadIdx.x;
  if (c >= chunks) return;
  const size_t row4 = (size_t)blockIdx.x * 4 * D * 2, row1 = (size_t)blockIdx.x * D * 2;
  u32x4 v[9];
  for (int g = 0; g < 4; ++g) {
    v[g] = __builtin_nontemporal_load((const u32x4 *)(s + row4 + (size_t)g * D * 2) + c);
    v[4 + g] = __builtin_nontemporal_load((const u32x4 *)(z + row4 + (size_t)g * D * 2) + c);
  }
  v[8] = __builtin_nontemporal_load((const u32x4 *)(pc + row1) + c);
  const u32x4 a = v[0] ^ v[1] ^ v[2] ^ v[3] ^ v[8], b = v[4] ^ v[5] ^ v[6] ^ v[7];
  __builtin_nontemporal_store(a, (u32x4 *)(out_cell + row1) + c);
  __builtin_nontemporal_store(b, (u32x4 *)(out_state + row1) + c);
}

// The same traffic requested the way the library's staged sum_lstm kernel requests it: cell gate; wait for it; forget
// gate's s; barrier; rest of the forget gate, previous cell, input gate; wait for forget gate and cell; output gate;
// wait for the input gate; store the cell; barrier; wait for the output gate; store the state.  No arithmetic: what
// the stages and their waits cost by themselves.
__global__ void lstm_traffic_staged_kernel(const char *s, const char *z, const char *pc, char *out_state,
                                           char *out_cell, int D) {
  const int c = threadIdx.x;   // the host launches D / 8 lanes, a multiple of 64
  const size_t row4 = (size_t)blockIdx.x * 4 * D * 2, row1 = (size_t)blockIdx.x * D * 2, gate = (size_t)D * 2;
  auto ld = [&](const char *p) { return __builtin_nontemporal_load((const u32x4 *)p + c); };
  const u32x4 zc = ld(z + row4 + 3 * gate), sc = ld(s + row4 + 3 * gate);
  __builtin_amdgcn_sched_barrier(0);
  u32x4 acc = zc ^ sc;
  __builtin_amdgcn_sched_barrier(0);
  const u32x4 sf = ld(s + row4);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  const u32x4 zf = ld(z + row4), cell = ld(pc + row1), si = ld(s + row4 + gate), zi = ld(z + row4 + gate);
  __builtin_amdgcn_sched_barrier(0);
  acc ^= sf ^ zf ^ cell;
  __builtin_amdgcn_sched_barrier(0);
  const u32x4 so = ld(s + row4 + 2 * gate), zo = ld(z + row4 + 2 * gate);
  __builtin_amdgcn_sched_barrier(0);
  acc ^= si ^ zi;
  __builtin_nontemporal_store(acc, (u32x4 *)(out_cell + row1) + c);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  __builtin_nontemporal_store(acc ^ so ^ zo, (u32x4 *)(out_state + row1) + c);
}

__global__ void ln_traffic_kernel(const char *x, char *out, int hidden) {
  const int c = threadIdx.x;
  if (c >= hidden / 8) return;
  const size_t row = (size_t)blockIdx.x * hidden * 2;
  const u32x4 v = __builtin_nontemporal_load((const u32x4 *)(x + row) + c);
  __builtin_nontemporal_store(v, (u32x4 *)(out + row) + c);
}

struct Three {
  char *p[3];
};

// mode 0: load 64 KiB pieces; 1: store 64 KiB pieces; 2: load 64 KiB, store 32 KiB; 3: load 64 KiB, store 32 KiB as 32
// rows of 1 KiB scattered over the destination - the bulk KV write's pattern, contiguous K/V rows in and random
// 1 KiB cache rows out.  Row g of the stream goes to the row whose low `scatter_bits` bits are those of g times an
// odd constant (a permutation of every aligned group of 2^scatter_bits rows; the host passes the number of trailing
// zero bits of the row count).
__global__ void stream_kernel(Three src, int nsrc, Three dst, int ndst, int64_t pieces, int mode, int scatter_bits,
                              unsigned *sink) {
  unsigned acc = 0;
  for (int64_t k = blockIdx.x; k < pieces; k += gridDim.x) {
    const u32x4 *from = (const u32x4 *)(src.p[k % nsrc] + (k / nsrc) * 65536);
    if (mode == 4) {
      // as mode 3 with 16-byte stores: a lane takes two adjacent 16-byte loads
      for (int i = threadIdx.x; i < 2048; i += blockDim.x) {
        const u32x4 v = __builtin_nontemporal_load(from + 2 * i), v2 = __builtin_nontemporal_load(from + 2 * i + 1);
        const u32x4 w = {v.x ^ v.z, v.y ^ v.w, v2.x ^ v2.z, v2.y ^ v2.w};
        const unsigned g = (unsigned)k * 32u + (unsigned)i / 64u, mask = (1u << scatter_bits) - 1u;
        const unsigned row = (g & ~mask) | ((g * 40503u) & mask);
        __builtin_nontemporal_store(w, (u32x4 *)(dst.p[row % ndst] + (row / ndst) * 1024) + i % 64);
      }
      continue;
    }
    for (int i = threadIdx.x; i < 4096; i += blockDim.x) {
      u32x4 v = {1u, 2u, 3u, (unsigned)i};
      if (mode != 1) v = __builtin_nontemporal_load(from + i);
      if (mode == 0) acc ^= v.x ^ v.y ^ v.z ^ v.w;
      if (mode == 1) __builtin_nontemporal_store(v, (u32x4 *)(dst.p[k % ndst] + (k / ndst) * 65536) + i);
      if (mode == 2) {
        const u32x2 w = {v.x ^ v.z, v.y ^ v.w};
        __builtin_nontemporal_store(w, (u32x2 *)(dst.p[k % ndst] + (k / ndst) * 32768) + i);
      }
      if (mode == 3) {
        const u32x2 w = {v.x ^ v.z, v.y ^ v.w};
        const unsigned g = (unsigned)k * 32u + (unsigned)i / 128u, mask = (1u << scatter_bits) - 1u;
        const unsigned row = (g & ~mask) | ((g * 40503u) & mask);
        __builtin_nontemporal_store(w, (u32x2 *)(dst.p[row % ndst] + (row / ndst) * 1024) + i % 128);
      }
    }
  }
  if (mode == 0 && acc == 0x12345677u) *sink = acc;
}

// The 2:1 stream with scattered 1 KiB rows (mode 3 of stream_kernel) by resident workgroups: a piece is kLoads x 16 KiB,
// every lane requests its kLoads chunks of it at once, then stores the halves; the rows are dealt over `ndst` buffers.
// period > 0: time slices.  Every workgroup requests its loads only while the shared 100 MHz clock, modulo `period`
// ticks, is below `read_ticks`, and stores only in the rest of the period, so that the memory system sees reads and
// writes in turns instead of mixed.  (Both waits end by themselves: the clock runs on.)
template <int kLoads>
__global__ __launch_bounds__(1024) void resident_stream_kernel(const char *src, Three dst, int ndst, int64_t pieces,
                                                                int scatter_bits, int period, int read_ticks) {
  const unsigned rows_per_piece = kLoads * 8;
  for (int64_t k = blockIdx.x; k < pieces; k += gridDim.x) {
    if (period > 0)
      while ((int)(wall_clock64() % (unsigned long long)period) >= read_ticks) __builtin_amdgcn_s_sleep(4);
    const u32x4 *from = (const u32x4 *)(src + k * (int64_t)kLoads * 16384);
    u32x4 v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) v[u] = __builtin_nontemporal_load(from + u * 1024 + threadIdx.x);
    if (period > 0) {
      if (v[kLoads - 1].x == 0x9e3779b9u && v[0].y == 0x12345u) __builtin_amdgcn_s_sleep(1);   // the data has arrived
      while ((int)(wall_clock64() % (unsigned long long)period) < read_ticks) __builtin_amdgcn_s_sleep(4);
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const u32x2 w = {v[u].x ^ v[u].z, v[u].y ^ v[u].w};
      const unsigned i = u * 1024 + threadIdx.x;
      const unsigned g = (unsigned)k * rows_per_piece + i / 128u, mask = (1u << scatter_bits) - 1u;
      const unsigned row = (g & ~mask) | ((g * 40503u) & mask);
      __builtin_nontemporal_store(w, (u32x2 *)(dst.p[row % ndst] + (int64_t)(row / ndst) * 1024) + i % 128);
    }
  }
}

// bytes_in of `src` (a multiple of loads x 16 KiB, at most 2^41) are read, half as many written, dealt over dst[0..ndst);
// period_ticks = 0: no time slices, else 0 < read_ticks < period_ticks (ticks of 10 ns)
// The traffic of the fp4 cache write and nothing else: one lane per group of 16 bf16 elements (the slot and two
// 16-byte loads requested together, then 8 bytes of packed values and one scale byte stored at the slot's row of
// contiguous caches).  `row_groups` = groups per token row (heads x head_size / 16); lanes walk a token's K row, then
// its V row.
__global__ __launch_bounds__(64) void fp4_traffic_kernel(const char *key, const char *value, char *key_cache,
                                                         char *value_cache, char *key_scales, char *value_scales,
                                                         const long long *slots, long long total_groups, int row_groups) {
  const long long idx = (long long)blockIdx.x * 64 + threadIdx.x;
  const long long at = idx < total_groups ? idx : total_groups - 1;
  const long long row = at / row_groups;
  const int in_row = (int)(at - row * row_groups);
  const long long token = row >> 1;
  const long long slot = slots[token];
  const char *src = ((row & 1) ? value : key) + (token * row_groups + in_row) * 32;
  const u32x4 lo = __builtin_nontemporal_load((const u32x4 *)src);
  const u32x4 hi = __builtin_nontemporal_load((const u32x4 *)(src + 16));
  __builtin_amdgcn_sched_barrier(0);
  if (idx >= total_groups || slot < 0) return;
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  const u32x2 packed = {lo.x ^ hi.x ^ lo.z ^ hi.z, lo.y ^ hi.y ^ lo.w ^ hi.w};
  __builtin_nontemporal_store(packed, (u32x2 *)(((row & 1) ? value_cache : key_cache) + (slot * row_groups + in_row) * 8));
  ((row & 1) ? value_scales : key_scales)[slot * row_groups + in_row] = (char)(packed.x >> 7);
}

extern "C" int floor_stream_resident(const void *src, void *const *dst, int ndst, int64_t bytes_in, int loads,
                                     int workgroups, int period_ticks, int read_ticks, void *stream) {
  if (!src || !dst || ndst < 1 || ndst > 3 || (loads != 4 && loads != 8) || workgroups < 1 || workgroups > 65535 ||
      bytes_in <= 0 || bytes_in % ((int64_t)loads * 16384) || bytes_in > ((int64_t)1 << 41))
    return 1;
  if (period_ticks < 0 || (period_ticks > 0 && (read_ticks <= 0 || read_ticks >= period_ticks))) return 1;
  Three d = {};
  for (int i = 0; i < ndst; ++i) d.p[i] = (char *)dst[i];
  const int64_t pieces = bytes_in / ((int64_t)loads * 16384);
  const int scatter_bits = __builtin_ctzll((unsigned long long)(pieces * loads * 8));
  hipStream_t s = (hipStream_t)stream;
  if (loads == 4)
    hipLaunchKernelGGL(resident_stream_kernel<4>, dim3(workgroups), dim3(1024), 0, s, (const char *)src, d, ndst, pieces, scatter_bits,
                       period_ticks, read_ticks);
  else
    hipLaunchKernelGGL(resident_stream_kernel<8>, dim3(workgroups), dim3(1024), 0, s, (const char *)src, d, ndst, pieces, scatter_bits,
                       period_ticks, read_ticks);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// Issue rates of the vector ALU: every lane runs `iters` rounds of eight independent chains of one operation
// (0 multiply, 1 fused multiply-add, 2 reciprocal, 3 exp2, 4 one reciprocal followed by three dependent full-rate
// operations, 5 16-bit unpack by shift, 6 v_cvt_f64_f32 . v_mul_f64 . v_cvt_f32_f64, 7 v_med3_f32).  The host times
// it with 1, 2 and 4 waves per SIMD.
template <int OP>
__global__ __launch_bounds__(256) void valu_rate_kernel(float *out, int iters, float seed) {
  float a[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) a[j] = seed + threadIdx.x * 1e-3f + j;
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (OP == 0) a[j] = a[j] * 1.0001f;
      if (OP == 1) a[j] = __builtin_fmaf(a[j], 1.0001f, 0.5f);
      if (OP == 2) a[j] = __builtin_amdgcn_rcpf(a[j]);
      if (OP == 3) a[j] = __builtin_amdgcn_exp2f(a[j]);
      if (OP == 4) {
        a[j] = __builtin_amdgcn_rcpf(a[j]);
        a[j] = a[j] * 1.0001f;
        a[j] = a[j] + 0.25f;
        a[j] = a[j] * a[j];
      }
      if (OP == 5) a[j] = __uint_as_float(__float_as_uint(a[j]) << 1);
      // the bulk write's exact division by the scale: widen, multiply in fp64, narrow (3 instructions per round)
      if (OP == 6) a[j] = (float)((double)a[j] * 1.0000001);
      if (OP == 7) a[j] = __builtin_amdgcn_fmed3f(a[j], -448.0f, 448.0f);
    }
  }
  float s = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += a[j];
  if (s == 123.456f) out[0] = s;   // never true: keeps the chains alive
}

// `blocks` workgroups of 256 lanes (one wave per SIMD of a CU each); returns 0 or an error code.
extern "C" int floor_valu_rate(int op, int blocks, int iters, void *out, void *stream) {
  if (blocks <= 0 || iters <= 0 || !out) return 1;
  const dim3 g((unsigned)blocks), b(256);
  hipStream_t s = (hipStream_t)stream;
  switch (op) {
    case 0: hipLaunchKernelGGL(valu_rate_kernel<0>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 1: hipLaunchKernelGGL(valu_rate_kernel<1>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 2: hipLaunchKernelGGL(valu_rate_kernel<2>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 3: hipLaunchKernelGGL(valu_rate_kernel<3>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 4: hipLaunchKernelGGL(valu_rate_kernel<4>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 5: hipLaunchKernelGGL(valu_rate_kernel<5>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 6: hipLaunchKernelGGL(valu_rate_kernel<6>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    case 7: hipLaunchKernelGGL(valu_rate_kernel<7>, g, b, 0, s, (float *)out, iters, 1.5f); break;
    default: return 1;
  }
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// What a kernel node costs when it moves (almost) nothing: `touch` = 0 an empty kernel, 1 one 16-byte load and one
// 16-byte store per lane of the first wave of every workgroup (a first byte's round trip, no bandwidth).
__global__ void node_floor_kernel(const u32x4 *in, u32x4 *out, int touch) {
  if (touch && threadIdx.x < 64) out[blockIdx.x * 64 + threadIdx.x] = in[blockIdx.x * 64 + threadIdx.x];
}

// in / out: blocks * 1 KiB each
extern "C" int floor_node(const void *in, void *out, int blocks, int threads, int touch, void *stream) {
  if (blocks <= 0 || threads < 64 || threads > 1024) return 1;
  hipLaunchKernelGGL(node_floor_kernel, dim3((unsigned)blocks), dim3((unsigned)threads), 0, (hipStream_t)stream,
                     (const u32x4 *)in, (u32x4 *)out, touch);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// The loads of the row-argmax kernel and nothing else: one workgroup per row, 16-byte streaming loads in batches of
// four per lane, the words xor-ed together.
__global__ __launch_bounds__(1024) void row_read_kernel(const char *in, int64_t row_bytes, unsigned *sink) {
  const u32x4 *row = (const u32x4 *)(in + (int64_t)blockIdx.x * row_bytes);
  const int chunks = (int)(row_bytes / 16);
  unsigned acc = 0;
  for (int c0 = threadIdx.x; c0 < chunks; c0 += 4 * blockDim.x) {
    u32x4 raw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (c0 + u * (int)blockDim.x < chunks) raw[u] = __builtin_nontemporal_load(row + c0 + u * blockDim.x);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (c0 + u * (int)blockDim.x < chunks) acc ^= raw[u].x ^ raw[u].y ^ raw[u].z ^ raw[u].w;
  }
  if (acc == 0x12345677u) *sink = acc;
}

extern "C" int floor_row_read(const void *in, int64_t rows, int64_t row_bytes, int threads, void *sink, void *stream) {
  if (rows <= 0 || row_bytes <= 0 || row_bytes % 16 != 0 || threads < 64 || threads > 1024 || !sink) return 1;
  hipLaunchKernelGGL(row_read_kernel, dim3((unsigned)rows), dim3((unsigned)threads), 0, (hipStream_t)stream,
                     (const char *)in, row_bytes, (unsigned *)sink);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

extern "C" int floor_ln_traffic(const void *x, void *out, int64_t rows, int hidden, void *stream) {
  if (hidden % 8 || hidden / 8 > 1024 || rows <= 0) return 1;
  hipLaunchKernelGGL(ln_traffic_kernel, dim3((unsigned)rows), dim3((unsigned)((hidden / 8 + 63) & ~63)), 0,
                     (hipStream_t)stream, (const char *)x, (char *)out, hidden);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

extern "C" int floor_lstm_traffic(const void *s, const void *z, const void *pc, void *out_state, void *out_cell,
                                  int64_t rows, int D, void *stream) {
  if (rows <= 0 || D <= 0 || D % 8 != 0 || D / 8 > 1024) return 1;
  hipLaunchKernelGGL(lstm_traffic_kernel, dim3((unsigned)rows), dim3((unsigned)((D / 8 + 63) & ~63)), 0,
                     (hipStream_t)stream, (const char *)s, (const char *)z, (const char *)pc, (char *)out_state,
                     (char *)out_cell, D);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

extern "C" int floor_fp4_traffic(const void *key, const void *value, void *key_cache, void *value_cache, void *key_scales,
                                 void *value_scales, const void *slots, long long num_tokens, int row_groups, void *stream) {
  if (num_tokens <= 0 || row_groups <= 0) return 1;
  const long long total = num_tokens * 2 * row_groups;
  if ((total + 63) / 64 > 0x7fffffffLL) return 1;
  hipLaunchKernelGGL(fp4_traffic_kernel, dim3((unsigned)((total + 63) / 64)), dim3(64), 0, (hipStream_t)stream,
                     (const char *)key, (const char *)value, (char *)key_cache, (char *)value_cache, (char *)key_scales,
                     (char *)value_scales, (const long long *)slots, total, row_groups);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

extern "C" int floor_lstm_traffic_staged(const void *s, const void *z, const void *pc, void *out_state, void *out_cell,
                                         int64_t rows, int D, void *stream) {
  if (rows <= 0 || D <= 0 || D % 512 != 0 || D / 8 > 1024) return 1;
  hipLaunchKernelGGL(lstm_traffic_staged_kernel, dim3((unsigned)rows), dim3((unsigned)(D / 8)), 0, (hipStream_t)stream,
                     (const char *)s, (const char *)z, (const char *)pc, (char *)out_state, (char *)out_cell, D);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// Each buffer must hold ceil(pieces / n) * 64 KiB.  `sink` is 4 bytes of device memory.
extern "C" int floor_stream(void *const *src, int nsrc, void *const *dst, int ndst, int64_t pieces, int mode,
                            void *sink, void *stream) {
  if (nsrc < 1 || nsrc > 3 || ndst < 1 || ndst > 3 || pieces <= 0 || mode < 0 || mode > 4 || !sink) return 1;
  Three a = {}, b = {};
  for (int i = 0; i < nsrc; ++i) a.p[i] = (char *)src[i];
  for (int i = 0; i < ndst; ++i) b.p[i] = (char *)dst[i];
  if (mode >= 3 && pieces * 32 >= (1LL << 31)) return 1;
  const int scatter_bits = __builtin_ctzll((unsigned long long)(pieces * 32));
  hipLaunchKernelGGL(stream_kernel, dim3(8192), dim3(256), 0, (hipStream_t)stream, a, nsrc, b, ndst, pieces, mode,
                     scatter_bits, (unsigned *)sink);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// The bulk write as the reference decomposes it (csrc/custom_ops/reshape_and_cache_flash_bulk.cu:12-60): one workgroup
// per (layer, token) of min(n, 512) lanes; a lane moves one element per step - a 2-byte load of K and of V, an fp32
// division by the layer's scale, a conversion, a 1-byte store each - and finds its place in the cache row with a
// division and a remainder by head_size per element; the slot, the two cache pointers and the two scale pointers are
// read from device memory by every workgroup.  bf16 source, e4m3 cache.  Same bytes out as the library's kernel
// (bench.py compares them); a measurement aid, not a code path of the package.
__device__ __forceinline__ unsigned char e4m3_of(float q) {
  if (q != q) return (unsigned char)(0x7fu | ((__float_as_uint(q) >> 24) & 0x80u));
  const float c = __builtin_amdgcn_fmed3f(q, -448.0f, 448.0f);
  return (unsigned char)(__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xff);
}

__global__ void write_per_layer_and_token_kernel(const unsigned short *keys, const unsigned short *values,
                                                 const int64_t *key_cache_ptrs, const int64_t *value_cache_ptrs,
                                                 const int64_t *slot_mapping, int64_t block_stride, int64_t key_stride,
                                                 int64_t value_stride, int num_heads, int head_size, int block_size,
                                                 const int64_t *k_scale_ptrs, const int64_t *v_scale_ptrs) {
  const int64_t layer = blockIdx.x, token = blockIdx.y;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;   // a padding token
  const int64_t block = slot / block_size, in_block = slot % block_size;
  const int n = num_heads * head_size;
  unsigned char *key_cache = (unsigned char *)key_cache_ptrs[layer];
  unsigned char *value_cache = (unsigned char *)value_cache_ptrs[layer];
  const float *k_scale = (const float *)k_scale_ptrs[layer];
  const float *v_scale = (const float *)v_scale_ptrs[layer];
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int head = i / head_size, in_head = i % head_size;
    const int64_t dst = block * block_stride + in_block * n + (int64_t)head * head_size + in_head;
    const float k = __uint_as_float((unsigned)keys[token * key_stride + layer * n + i] << 16);
    const float v = __uint_as_float((unsigned)values[token * value_stride + layer * n + i] << 16);
    key_cache[dst] = e4m3_of(k / *k_scale);
    value_cache[dst] = e4m3_of(v / *v_scale);
  }
}

// The four pointer tables are int64[num_layers] in DEVICE memory (the reference's launcher copies them there on
// every call, :104-131).  Strides in elements.
extern "C" int floor_write_per_layer_and_token(const void *keys, const void *values, const void *key_cache_ptrs,
                                               const void *value_cache_ptrs, const void *slot_mapping,
                                               int64_t num_tokens, int num_layers, int64_t block_stride,
                                               int64_t key_stride, int64_t value_stride, int num_heads, int head_size,
                                               int block_size, const void *k_scale_ptrs, const void *v_scale_ptrs,
                                               void *stream) {
  if (num_tokens <= 0 || num_tokens > 65535 || num_layers <= 0 || num_heads <= 0 || head_size <= 0 || block_size <= 0 ||
      (int64_t)num_heads * head_size > (1 << 24))
    return 1;
  const int n = num_heads * head_size;
  hipLaunchKernelGGL(write_per_layer_and_token_kernel, dim3((unsigned)num_layers, (unsigned)num_tokens),
                     dim3((unsigned)(n < 512 ? n : 512)), 0, (hipStream_t)stream, (const unsigned short *)keys,
                     (const unsigned short *)values, (const int64_t *)key_cache_ptrs, (const int64_t *)value_cache_ptrs,
                     (const int64_t *)slot_mapping, block_stride, key_stride, value_stride, num_heads, head_size,
                     block_size, (const int64_t *)k_scale_ptrs, (const int64_t *)v_scale_ptrs);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// eight bf16 elements of a row, stored through the caches (both decompositions below read a row again)
__device__ __forceinline__ void store8(char *row, int chunk, const float (&f)[8]) {
  const uint4 v = arctic::pack8<arctic::BF16>(f);
  const arctic::u32x4 words = {v.x, v.y, v.z, v.w};
  *(ARCTIC_GLOBAL arctic::u32x4 *)(row + (int64_t)chunk * 16) = words;
}

// sum_lstm as the reference decomposes it (csrc/custom_ops/sum_lstm.cu:28-191): one workgroup of 128 lanes per row,
// 16 bytes per lane and step, and three passes over global memory - the cell's pre-activation alone for its sum of
// squares; then the forget, input and cell pre-activations with the previous cell, for the new cell, which is stored;
// then the stored cell read back, with the output gate's pre-activation, for the state - with a block-wide sum after
// each of the first two, and sigmoid and GELU through the C library's expf and erff.  bf16, all four vectors given.
// Results agree with the library's kernel within the operators' tolerance (bench.py checks); a measurement aid.
namespace three_passes {

constexpr int kLanes = 128;

__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f)); }

__device__ __forceinline__ void load8(const char *p, int chunk, float (&f)[8]) {
  arctic::Chunk::load(p + (int64_t)chunk * 16).unpack<arctic::BF16>(f);
}
// s + alpha * z of gate g (0 forget, 1 input, 2 output, 3 cell), chunk i
__device__ __forceinline__ void pre_activation(const char *s, const char *z, int64_t gate_bytes, int g, int i,
                                               float alpha, float (&f)[8]) {
  float a[8], b[8];
  load8(s + g * gate_bytes, i, a);
  load8(z + g * gate_bytes, i, b);
#pragma unroll
  for (int k = 0; k < 8; ++k) f[k] = a[k] + alpha * b[k];
}

__global__ __launch_bounds__(kLanes) void sum_lstm_kernel(char *out_state, char *out_cell, const char *states,
                                                          const char *z4, const char *prev_cell, const char *w_cell,
                                                          const char *b_cell, const char *w_state, const char *b_state,
                                                          int64_t s_pitch, int64_t z_pitch, int64_t c_pitch,
                                                          int64_t o_pitch, int D, float alpha, float eps_cell,
                                                          float eps_state) {
  typedef hipcub::BlockReduce<float, kLanes> Reduce;
  __shared__ typename Reduce::TempStorage scratch0, scratch1;
  __shared__ float inv_rms_pre, inv_rms_cell;
  const int64_t row = blockIdx.x;
  const char *s = states + row * s_pitch, *z = z4 + row * z_pitch, *pc = prev_cell + row * c_pitch;
  char *cell_row = out_cell + row * o_pitch, *state_row = out_state + row * o_pitch;
  const int chunks = D / 8;
  const int64_t gate_bytes = (int64_t)D * 2;

  float ss = 0.f;
  for (int i = threadIdx.x; i < chunks; i += kLanes) {
    float c[8];
    pre_activation(s, z, gate_bytes, 3, i, alpha, c);
#pragma unroll
    for (int k = 0; k < 8; ++k) ss += c[k] * c[k];
  }
  float total = Reduce(scratch0).Sum(ss);
  if (threadIdx.x == 0) inv_rms_pre = rsqrtf(total / (float)D + eps_cell);
  __syncthreads();

  ss = 0.f;
  for (int i = threadIdx.x; i < chunks; i += kLanes) {
    float f[8], in[8], c[8], p[8], w[8], b[8], cell[8];
    pre_activation(s, z, gate_bytes, 0, i, alpha, f);
    pre_activation(s, z, gate_bytes, 1, i, alpha, in);
    pre_activation(s, z, gate_bytes, 3, i, alpha, c);
    load8(pc, i, p);
    load8(w_cell, i, w);
    load8(b_cell, i, b);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      float normed = c[k] * inv_rms_pre;
      normed *= w[k];
      normed += b[k];
      cell[k] = p[k] * sigmoid(f[k]) + gelu(normed) * sigmoid(in[k]);
      ss += cell[k] * cell[k];
    }
    store8(cell_row, i, cell);
  }
  total = Reduce(scratch1).Sum(ss);
  if (threadIdx.x == 0) inv_rms_cell = rsqrtf(total / (float)D + eps_state);
  __syncthreads();

  for (int i = threadIdx.x; i < chunks; i += kLanes) {
    float c[8], o[8], w[8], b[8], state[8];
    load8(cell_row, i, c);   // the rounded cell this lane stored above
    pre_activation(s, z, gate_bytes, 2, i, alpha, o);
    load8(w_state, i, w);
    load8(b_state, i, b);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      float normed = c[k] * inv_rms_cell;
      normed *= w[k];
      normed += b[k];
      state[k] = gelu(normed) * sigmoid(o[k]);
    }
    store8(state_row, i, state);
  }
}

}  // namespace three_passes

// bf16 rows; pitches in elements; D a multiple of 8; every pointer 16-byte aligned and none null.
extern "C" int floor_sum_lstm_three_passes(void *out_state, void *out_cell, const void *states, const void *z4,
                                           const void *prev_cell, const void *w_cell, const void *b_cell,
                                           const void *w_state, const void *b_state, int64_t rows, int D, int64_t s_pitch,
                                           int64_t z_pitch, int64_t c_pitch, int64_t o_pitch, float alpha, float eps_cell,
                                           float eps_state, void *stream) {
  if (rows <= 0 || rows > 0x7fffffffLL || D <= 0 || D % 8 || (s_pitch | z_pitch | c_pitch | o_pitch) % 8) return 1;
  const void *all[9] = {out_state, out_cell, states, z4, prev_cell, w_cell, b_cell, w_state, b_state};
  for (const void *p : all)
    if (!p || ((uintptr_t)p & 15)) return 1;
  hipLaunchKernelGGL(three_passes::sum_lstm_kernel, dim3((unsigned)rows), dim3(three_passes::kLanes), 0,
                     (hipStream_t)stream, (char *)out_state, (char *)out_cell, (const char *)states, (const char *)z4,
                     (const char *)prev_cell, (const char *)w_cell, (const char *)b_cell, (const char *)w_state,
                     (const char *)b_state, s_pitch * 2, z_pitch * 2, c_pitch * 2, o_pitch * 2, D, alpha, eps_cell,
                     eps_state);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}

// speculator_ln as the reference decomposes it (csrc/custom_ops/speculator_ln.cu:21-107; 256 lanes per row from 256
// rows on, :203-207): a first pass over the row for its sum of squares, a block sum, a second pass that reads the row
// again, scales it, applies weight and bias and stores.  bf16, weight and bias given, output rows dense.
namespace two_passes {

constexpr int kLanes = 256;

__global__ __launch_bounds__(kLanes) void ln_kernel(char *out, const char *in, const char *weight, const char *bias,
                                                    int64_t in_pitch, int hidden, float eps) {
  typedef hipcub::BlockReduce<float, kLanes> Reduce;
  __shared__ typename Reduce::TempStorage scratch;
  __shared__ float inv_rms;
  const char *row_in = in + (int64_t)blockIdx.x * in_pitch;
  char *row_out = out + (int64_t)blockIdx.x * hidden * 2;
  const int chunks = hidden / 8;
  float ss = 0.f;
  for (int i = threadIdx.x; i < chunks; i += kLanes) {
    float x[8];
    three_passes::load8(row_in, i, x);
#pragma unroll
    for (int k = 0; k < 8; ++k) ss += x[k] * x[k];
  }
  const float total = Reduce(scratch).Sum(ss);
  if (threadIdx.x == 0) inv_rms = rsqrtf(total / (float)hidden + eps);
  __syncthreads();
  for (int i = threadIdx.x; i < chunks; i += kLanes) {
    float x[8], w[8], b[8], y[8];
    three_passes::load8(row_in, i, x);
    three_passes::load8(weight, i, w);
    three_passes::load8(bias, i, b);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      y[k] = x[k] * inv_rms;
      y[k] *= w[k];
      y[k] += b[k];
    }
    store8(row_out, i, y);
  }
}

}  // namespace two_passes

// bf16; in_pitch in elements; hidden a multiple of 8; every pointer 16-byte aligned and none null.
extern "C" int floor_ln_two_passes(void *out, const void *in, const void *weight, const void *bias, int64_t rows,
                                   int hidden, int64_t in_pitch, float eps, void *stream) {
  if (rows <= 0 || rows > 0x7fffffffLL || hidden <= 0 || hidden % 8 || in_pitch % 8) return 1;
  const void *all[4] = {out, in, weight, bias};
  for (const void *p : all)
    if (!p || ((uintptr_t)p & 15)) return 1;
  hipLaunchKernelGGL(two_passes::ln_kernel, dim3((unsigned)rows), dim3(two_passes::kLanes), 0, (hipStream_t)stream,
                     (char *)out, (const char *)in, (const char *)weight, (const char *)bias, in_pitch * 2, hidden, eps);
  return hipGetLastError() == hipSuccess ? 0 : 3;
}
