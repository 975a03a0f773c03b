// Device helpers shared by the kernel translation units of libstile_hip.so.
#pragma once

#include "stile_internal.h"

#include <hip/hip_bf16.h>

#include <type_traits>

namespace stile {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4 ld4(const float* p) {
  return *reinterpret_cast<const float4*>(p);
}
__device__ __forceinline__ void st4(float* p, float4 v) {
  *reinterpret_cast<float4*>(p) = v;
}
__device__ __forceinline__ float comp(const float4& v, int t) {
  return t == 0 ? v.x : (t == 1 ? v.y : (t == 2 ? v.z : v.w));
}

// Neumaier compensated accumulation: s + c carries the sum of every x added.
// Contraction is off so (s - t) + x is evaluated as written.
__device__ __forceinline__ void neu_add(float& s, float& c, float x) {
#pragma clang fp contract(off)
  float t = s + x;
  if (fabsf(s) >= fabsf(x))
    c += (s - t) + x;
  else
    c += (x - t) + s;
  s = t;
}

// Elements of B: FP32, BF16 or FP16.  load_b4 returns four consecutive
// columns of row k starting at column col as FP32 (exact for the 16-bit
// types); columns at or beyond N read as 0.  vec: B rows are aligned for one
// vector load of four elements (16 bytes FP32, 8 bytes 16-bit) and N % 4 == 0.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

template <typename TB>
__device__ __forceinline__ float4 cvt4(uint2 w) {
  if constexpr (std::is_same<TB, __bf16>::value) {
    return make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
  } else {
    const f16x2 a = __builtin_bit_cast(f16x2, w.x), b = __builtin_bit_cast(f16x2, w.y);
    return make_float4((float)a[0], (float)a[1], (float)b[0], (float)b[1]);
  }
}

// B[k][col .. col + 3] as float4, zero at or beyond N.  vec (N % 4 == 0,
// rows aligned): one unconditional load from a column clamped into the row
// and a select after it.  (A load under an exec mask leaves its registers
// partly unwritten, and the compiler then waits for every load in flight
// before it reuses them: in a loop of gathers that serialises the gathers.)
template <typename TB>
__device__ __forceinline__ float4 load_b4(const TB* __restrict__ B, int64_t ldb, int k, int col, int N, bool vec) {
  const TB* p = B + (int64_t)k * ldb + col;
  if (vec) {
    const TB* q = B + (int64_t)k * ldb + min(col, N - 4);
    float4 r;
    if constexpr (std::is_same<TB, float>::value)
      r = ld4(q);
    else
      r = cvt4<TB>(*reinterpret_cast<const uint2*>(q));
    return col < N ? r : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float4 r;
  r.x = col < N ? (float)p[0] : 0.f;
  r.y = col + 1 < N ? (float)p[1] : 0.f;
  r.z = col + 2 < N ? (float)p[2] : 0.f;
  r.w = col + 3 < N ? (float)p[3] : 0.f;
  return r;
}

// f(std::true_type) when vec, else f(std::false_type): the row gathers of
// the sparse kernels see vec as a constant, so the 16-byte and the
// per-element paths of load_b4 are not merged into one loop, where the
// per-element path's masked loads make every gather wait for the ones
// before it.
template <typename F>
__device__ __forceinline__ void with_vec(bool vec, F&& f) {
  if (vec)
    f(std::true_type{});
  else
    f(std::false_type{});
}

// NT: non-temporal store (streamed past the caches; for rows nothing reads
// back soon).
template <bool NT = false>
__device__ __forceinline__ void store_c4(float* __restrict__ C, int64_t ldc,
                                         int row, int col, int N, bool vec,
                                         float4 v) {
  float* p = C + (int64_t)row * ldc + col;
  if (vec) {
    if (col < N) {
      if constexpr (NT) {
        typedef float f32v4 __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(f32v4{v.x, v.y, v.z, v.w}, reinterpret_cast<f32v4*>(p));
      } else {
        st4(p, v);
      }
    }
    return;
  }
  if (col < N) p[0] = v.x;
  if (col + 1 < N) p[1] = v.y;
  if (col + 2 < N) p[2] = v.z;
  if (col + 3 < N) p[3] = v.w;
}

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  const uint16_t a = __builtin_bit_cast(uint16_t, (__bf16)lo);
  const uint16_t b = __builtin_bit_cast(uint16_t, (__bf16)hi);
  return (uint32_t)a | ((uint32_t)b << 16);
}

__device__ __forceinline__ uint32_t half_sel(uint32_t x, uint32_t y, int hi) {
  // (x.lo, y.lo) or (x.hi, y.hi) as one packed pair: one v_perm_b32, whose
  // selector bytes 0-3 pick bytes of its second operand (x), 4-7 of its
  // first (y)
  return __builtin_amdgcn_perm(y, x, hi ? 0x07060302u : 0x05040100u);
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 lds_u128;

__device__ __forceinline__ i16x4 lds_tr_read(lds_u8* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_i16x4*>(p));
}

}  // namespace stile
