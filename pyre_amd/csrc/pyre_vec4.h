// Four elements at a time for the row kernels and for whoever finishes a product's partial sums
// himself: loads and stores of four float32 or bfloat16 values, and the sum of a product's partial
// sums in their fixed order.
#pragma once

#include "pyre_common.h"

namespace pyre {

template <typename T> struct Vec4;
template <> struct Vec4<float> {
  static __device__ inline float4 load(const float* p) { return *reinterpret_cast<const float4*>(p); }
  static __device__ inline void store(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
};
template <> struct Vec4<bf16> {
  static __device__ inline float4 load(const bf16* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    float4 v;
    v.x = __uint_as_float(u.x << 16);
    v.y = __uint_as_float(u.x & 0xffff0000u);
    v.z = __uint_as_float(u.y << 16);
    v.w = __uint_as_float(u.y & 0xffff0000u);
    return v;
  }
  static __device__ inline void store(bf16* p, float4 v) {
    uint2 u;
    u.x = pack_bf16x2(v.x, v.y);
    u.y = pack_bf16x2(v.z, v.w);
    *reinterpret_cast<uint2*>(p) = u;
  }
};

// The same loads and stores past the caches, for rows that are read and written once in a step of
// many rows (more bytes than the caches hold). The row kernels take them from kStreamElements elements on: 16 MB of float32 (us a
// launch at 1,777 rows of 3,584, two partial sums: LayerNorm with its term's own norm 31.1 -> 25.4, sums of two terms with three norms
// 36 -> 31; two streams of 1,536 at 2,048 rows 18.0 -> 15.7 and at 952 rows, 12 MB, 10.8 -> 11.5; PolyNorm of 8,960 at 2,048 and 952
// rows 30.8 -> 22.0 and 16.5 -> 12.5).
constexpr long kStreamElements = 1L << 22;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
template <typename T> struct Stream4;
template <> struct Stream4<float> {
  static __device__ inline float4 load(const float* p) {
    const f32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
    return float4{v[0], v[1], v[2], v[3]};
  }
  static __device__ inline void store(float* p, float4 v) {
    __builtin_nontemporal_store(f32x4_t{v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4_t*>(p));
  }
};
template <> struct Stream4<bf16> {
  static __device__ inline float4 load(const bf16* p) {
    const u32x2_t u = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p));
    return float4{__uint_as_float(u[0] << 16), __uint_as_float(u[0] & 0xffff0000u), __uint_as_float(u[1] << 16),
                  __uint_as_float(u[1] & 0xffff0000u)};
  }
  static __device__ inline void store(bf16* p, float4 v) {
    __builtin_nontemporal_store(u32x2_t{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)}, reinterpret_cast<u32x2_t*>(p));
  }
};

__device__ inline float4 add4(float4 a, float4 b) { return float4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }

// p[0] + p[1] + ... + p[n - 1] (in that order) of the float4 at `src` in each of n partial sums that
// lie `stride` elements apart. Up to kAtOnce loads are in flight together: a kernel that only
// passes a few rows on spends its time waiting for loads, one round trip after the other.
constexpr int kAtOnce = 12;
// The loads and the sum apart, for whoever asks for something else between the two.
template <typename T>
struct PendingSum4 {
  float4 v[kAtOnce];
  __device__ inline void ask(const T* src, size_t stride, int n) {
#pragma unroll
    for (int p = 0; p < kAtOnce; ++p)
      if (p < n) v[p] = Vec4<T>::load(src + p * stride);
  }
  __device__ inline float4 sum(const T* src, size_t stride, int n) const {
    float4 s = v[0];
#pragma unroll
    for (int p = 1; p < kAtOnce; ++p)
      if (p < n) s = add4(s, v[p]);
    for (int p = kAtOnce; p < n; ++p) s = add4(s, Vec4<T>::load(src + p * stride));
    return s;
  }
};
template <typename T>
__device__ inline float4 sum_partials4(const T* src, size_t stride, int n) {
  PendingSum4<T> pending;
  pending.ask(src, stride, n);
  return pending.sum(src, stride, n);
}

// The same sum of loads past the caches, in the same order.
template <typename T>
__device__ inline float4 sum_partials4_stream(const T* src, size_t stride, int n) {
  float4 s = Stream4<T>::load(src);
  for (int p = 1; p < n; ++p) s = add4(s, Stream4<T>::load(src + p * stride));
  return s;
}
// Four of them under way at a time, for products in up to ten parts and more (rows in such numbers hide a trip through memory behind
// each other, not one for each part). Kernels with many registers that see one or two parts are slower with it (two streams of 1,536 at
// 2,048 rows 16.7 -> 18.9 us).
template <typename T>
__device__ inline float4 sum_many_partials4_stream(const T* src, size_t stride, int n) {
  float4 s = Stream4<T>::load(src);
  for (int p = 1; p < n; p += 4) {
    float4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (p + i < n) v[i] = Stream4<T>::load(src + (p + i) * stride);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (p + i < n) s = add4(s, v[i]);
  }
  return s;
}

}  // namespace pyre
