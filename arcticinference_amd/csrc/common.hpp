// Shared device helpers for the gfx950 kernels: 16-bit float conversion,
// 16-byte vector access, wave64 DPP reductions and the error channel of the C ABI.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/arctic_mi355x.h"

namespace arctic {

// ---- error channel ---------------------------------------------------------
int fail(int code, const char *fmt, ...);
int check_launch(const char *what);

// A row pitch (in elements) that `rows` rows of a tensor inside a 2^47-byte address space can have: not negative,
// and the last row's byte offset stays inside that space, so that no product of the two formed later, on the host
// or in a kernel, overflows 64 bits.
inline bool pitch_ok(int64_t pitch_elems, int64_t rows, int elem_bytes) {
  if (pitch_elems < 0) return false;
  const int64_t limit = ((int64_t)1 << 47) / elem_bytes;
  return pitch_elems <= limit / (rows > 1 ? rows - 1 : 1);
}

// Division of numbers below 2^31 by one that is known at launch: a product and a shift in place of the thirty (32 bits) to
// hundred (64 bits) instructions of a general division.  With s = ceil(log2 d) and m = floor(2^(31+s) / d) + 1, which is
// at most 2^32 - 1, m d - 2^(31+s) lies in (0, 2^s], so that m n / 2^(31+s) exceeds n / d by less than 1 / d for every
// n < 2^31 and has the same integer part.
struct Divisor {
  uint32_t m, shift, d;
  Divisor() = default;
  explicit Divisor(uint32_t by) : d(by) {
    uint32_t s = 0;
    while (((uint64_t)1 << s) < by) ++s;
    shift = 31 + s;
    m = (uint32_t)(((uint64_t)1 << shift) / by + 1);
  }
  __host__ __device__ uint32_t quotient(uint32_t n) const { return (uint32_t)(((uint64_t)n * m) >> shift); }
};

// A launch.  The host writes a launch's arguments into the GPU's memory, and what that costs is the processor's stores over
// the bus: an empty kernel with one structure of up to 112 bytes is issued in 2.4 to 2.8 us (two levels, by where the process
// runs), with one of 256 to 768 bytes in 2.5 to 3.5 us, with 2288 bytes in 2.6 to 3.8 us, and with ten scalars in place of a
// structure of 64 bytes in 2.5 to 3.3 us.  The kernels launched here (the cache writes in 16-byte accesses, the norm, the gate
// update, the argmax) therefore have one structure or two, as small as their contents allow, but for the tables of 64 layers
// that every selecting write carries, and none of them asks for blockDim or gridDim: for those the runtime appends 256 bytes.
// The structures go to the runtime from where they are, without the copy that passing them by value to the kernel's host-side
// function makes.  (The row gather, the row map and the element-wise cache write are launched the usual way.)
template <typename... Args>
inline void launch(void (*kernel)(Args...), dim3 grid, int lanes, hipStream_t s, const Args &...args) {
  void *list[] = {const_cast<Args *>(&args)...};
  (void)hipLaunchKernel((const void *)kernel, grid, dim3((unsigned)lanes), list, 0, s);   // check_launch() reports an error
}

// ---- 16-bit floats ---------------------------------------------------------
// Activation element types. to_float is exact; from_float rounds to nearest
// even (what __float2bfloat16 / __float2half do in the reference,
// csrc/custom_ops/dtype_common.cuh:13-35).
struct BF16 {
  static constexpr int kCode = ARCTIC_DTYPE_BF16;
  __device__ static __forceinline__ float lo(uint32_t w) {
    return __uint_as_float(w << 16);
  }
  __device__ static __forceinline__ float hi(uint32_t w) {
    return __uint_as_float(w & 0xffff0000u);
  }
  // gfx950 rounds fp32 pairs to bf16 in hardware (v_cvt_pk_bf16_f32, RNE)
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ uint32_t pack(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
  __device__ static __forceinline__ uint32_t round_bits(float f) { return pack(f, 0.f) & 0xffffu; }
  // value of the rounded 16-bit number, as fp32
  __device__ static __forceinline__ float requant(float f) {
    return __uint_as_float(pack(f, 0.f) << 16);
  }
};

struct F16 {
  static constexpr int kCode = ARCTIC_DTYPE_F16;
  __device__ static __forceinline__ float lo(uint32_t w) {
    return __half2float(__ushort_as_half((unsigned short)(w & 0xffffu)));
  }
  __device__ static __forceinline__ float hi(uint32_t w) {
    return __half2float(__ushort_as_half((unsigned short)(w >> 16)));
  }
  __device__ static __forceinline__ uint32_t round_bits(float f) {
    return (uint32_t)__half_as_ushort(__float2half_rn(f));
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) {
    return round_bits(a) | (round_bits(b) << 16);
  }
  __device__ static __forceinline__ float requant(float f) {
    return __half2float(__float2half_rn(f));
  }
};

// Eight 16-bit elements (one 16-byte lane access) unpacked to fp32 and back.
template <typename T>
__device__ __forceinline__ void unpack8(const uint4 &v, float (&f)[8]) {
  f[0] = T::lo(v.x);
  f[1] = T::hi(v.x);
  f[2] = T::lo(v.y);
  f[3] = T::hi(v.y);
  f[4] = T::lo(v.z);
  f[5] = T::hi(v.z);
  f[6] = T::lo(v.w);
  f[7] = T::hi(v.w);
}

template <typename T>
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  uint4 v;
  v.x = T::pack(f[0], f[1]);
  v.y = T::pack(f[2], f[3]);
  v.z = T::pack(f[4], f[5]);
  v.w = T::pack(f[6], f[7]);
  return v;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Every tensor on these paths lives in device (global) memory.  Saying so keeps
// the compiler from falling back to flat_* instructions when a pointer has been
// round-tripped through LDS or a struct.
#define ARCTIC_GLOBAL __attribute__((address_space(1)))

__device__ __forceinline__ uint4 load16(const void *p) {
  const u32x4 v = *(const ARCTIC_GLOBAL u32x4 *)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
// streaming (non-temporal) variants: every byte on these paths is touched exactly once
__device__ __forceinline__ uint4 load16_stream(const void *p) {
  const u32x4 v = __builtin_nontemporal_load((const ARCTIC_GLOBAL u32x4 *)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void store16_stream(void *p, const uint4 &v) {
  const u32x4 t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, (ARCTIC_GLOBAL u32x4 *)p);
}
__device__ __forceinline__ void store8_stream(void *p, const uint2 &v) {
  const u32x2 t = {v.x, v.y};
  __builtin_nontemporal_store(t, (ARCTIC_GLOBAL u32x2 *)p);
}
__device__ __forceinline__ void store4_stream(void *p, uint32_t v) {
  __builtin_nontemporal_store(v, (ARCTIC_GLOBAL uint32_t *)p);
}

// The same for addresses that are only element-aligned (rows of odd widths or pitches): still one 16-byte access per
// lane, which the memory pipeline takes at any alignment; a wave's accesses then touch one 128-byte line more.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
template <bool kAnyAlignment>
__device__ __forceinline__ uint4 load16(const void *p) {
  if constexpr (!kAnyAlignment) return load16(p);
  const u32x4 v = *(const ARCTIC_GLOBAL u32x4_any *)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool kAnyAlignment>
__device__ __forceinline__ uint4 load16_stream(const void *p) {
  if constexpr (!kAnyAlignment) return load16_stream(p);
  const u32x4 v = __builtin_nontemporal_load((const ARCTIC_GLOBAL u32x4_any *)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool kAnyAlignment>
__device__ __forceinline__ void store16_stream(void *p, const uint4 &v) {
  if constexpr (!kAnyAlignment) return store16_stream(p, v);
  const u32x4_any t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, (ARCTIC_GLOBAL u32x4_any *)p);
}

// A lane's unit of work on the speculator paths: eight consecutive 16-bit elements
// moved with one 16-byte access.  (8-byte units with twice the lanes took 512 rows of 4096 of the gate update in 10.7 us where
// these took 10.0, all requests at once; that is the only size they were timed at, few rows were not.)
struct Chunk {
  static constexpr int kElems = 8;
  static constexpr int kBytes = 16;
  uint4 v;
  __device__ static __forceinline__ Chunk zero() { return Chunk{make_uint4(0, 0, 0, 0)}; }
  template <bool kAnyAlignment = false>
  __device__ static __forceinline__ Chunk load(const void *p) { return Chunk{load16<kAnyAlignment>(p)}; }
  template <bool kAnyAlignment = false>
  __device__ static __forceinline__ Chunk load_stream(const void *p) { return Chunk{load16_stream<kAnyAlignment>(p)}; }
  template <bool kAnyAlignment = false>
  __device__ __forceinline__ void store_stream(void *p) const { store16_stream<kAnyAlignment>(p, v); }
  template <typename T>
  __device__ __forceinline__ void unpack(float (&f)[8]) const { unpack8<T>(v, f); }
  template <typename T>
  __device__ static __forceinline__ Chunk pack(const float (&f)[8]) { return Chunk{pack8<T>(f)}; }
};

// A row of any width from 8 elements on is covered by chunks of 8: chunk c starts at element 8 c, the last one at D - 8,
// so that it ends with the row.  Where the width is no multiple of 8 the last chunk's first elements are the end of the
// chunk before it: they are computed twice, bit for bit alike, stored twice and counted once.  `repeated` says how many
// of a chunk's elements do not count: 0, 1 to 7 in such a last chunk, 8 or more for a lane behind the row's end.
struct Place {
  uint32_t off;   // bytes from the row's start
  int repeated;
  Place() = default;
  __device__ __forceinline__ Place(int chunk, int D) {
    const int start = min(chunk * Chunk::kElems, D - Chunk::kElems);
    off = (uint32_t)start * 2;
    repeated = chunk * Chunk::kElems - start;
  }
  __device__ __forceinline__ bool live() const { return repeated < Chunk::kElems; }
};

// ---- wave64 / workgroup reductions ------------------------------------------
// DPP butterfly inside each row of 16 lanes, then the four row totals are read
// with v_readlane.  Every lane returns the same wave total.
template <int kCtrl>
__device__ __forceinline__ float dpp_add(float v) {
  int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true);
  return v + __int_as_float(moved);
}

__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  v = dpp_add<0x140>(v);  // row_mirror
  const int b = __float_as_int(v);
  float r0 = __int_as_float(__builtin_amdgcn_readlane(b, 0));
  float r1 = __int_as_float(__builtin_amdgcn_readlane(b, 16));
  float r2 = __int_as_float(__builtin_amdgcn_readlane(b, 32));
  float r3 = __int_as_float(__builtin_amdgcn_readlane(b, 48));
  return (r0 + r1) + (r2 + r3);
}

// Sum over the whole workgroup of `nwaves` full waves (at most 16).  `slots` is
// LDS for 16 floats, private to this call site.  Each wave
// leaves its total in slots[wave]; after the barrier every row of 16 lanes reads
// the 16 slots (zero beyond the last wave) and folds them with the same DPP
// butterfly, so all lanes of all waves end with the identical total and no loop
// or branch depends on the number of waves.  (The callers know the number of waves from their arguments: blockDim is
// among 256 bytes that the runtime appends to the arguments of a kernel that asks for it.)
__device__ __forceinline__ float block_sum(float v, float *slots, int nwaves) {
  v = wave_sum(v);
  if (nwaves == 1) return v;
  const int lane = threadIdx.x & 63;
  if (lane == 0) slots[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = ((lane & 15) < nwaves) ? slots[lane & 15] : 0.f;
  t = dpp_add<0xB1>(t);   // quad_perm [1,0,3,2]
  t = dpp_add<0x4E>(t);   // quad_perm [2,3,0,1]
  t = dpp_add<0x141>(t);  // row_half_mirror
  t = dpp_add<0x140>(t);  // row_mirror
  return t;
}

}  // namespace arctic
