// pk_tdt_math.h - arithmetic shared by the TDT decoder's kernels: the two
// execution profiles, the activations written out term for term, and the
// coherent accesses of values that workgroups exchange.
#ifndef PK_TDT_MATH_H
#define PK_TDT_MATH_H

#include "pk_internal.h"

#pragma clang fp contract(off)

namespace pk {
namespace {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

// W: weight and encoder-row element; W4: four weights (one 8- or 16-byte
// load); X: a chain input as staged in LDS; A4: four chain accumulators.
struct ProfileF16 {
  typedef _Float16 W;
  typedef half4 W4;
  typedef _Float16 X;
  typedef half4 A4;
};
struct ProfileF32 {
  typedef float W;
  typedef float4v W4;
  typedef float X;
  typedef float4v A4;
};

template <class P>
__device__ __forceinline__ const typename P::W* wptr(const void* p) {
  return static_cast<const typename P::W*>(p);
}

__device__ __forceinline__ float exp_f32(float x) {
  const float log2e = 1.44269502f;
  const float ln2_hi = 0.693145751953125f;
  const float ln2_lo = 1.42860682030941723212e-6f;
  const float n = __builtin_rintf(x * log2e);
  float r = __builtin_fmaf(-n, ln2_hi, x);
  r = __builtin_fmaf(-n, ln2_lo, r);
  float p = 1.0f / 5040.0f;
  p = __builtin_fmaf(p, r, 1.0f / 720.0f);
  p = __builtin_fmaf(p, r, 1.0f / 120.0f);
  p = __builtin_fmaf(p, r, 1.0f / 24.0f);
  p = __builtin_fmaf(p, r, 1.0f / 6.0f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  const int ni = (int)n;
  const float scale = __uint_as_float((uint32_t)(ni + 127) << 23);
  return p * scale;
}

__device__ __forceinline__ float tanh_f32(float x) {
  const float a = fabsf(x);
  const float t = 1.0f - 2.0f / (exp_f32(2.0f * a) + 1.0f);
  return x < 0.0f ? -t : t;
}

__device__ __forceinline__ float sigmoid_f32(float v) {
  const float bounded = fminf(fmaxf(v, -20.0f), 20.0f);
  return 1.0f / (1.0f + exp_f32(-bounded));
}

__device__ __forceinline__ float clamped_tanh(float v) { return tanh_f32(fminf(fmaxf(v, -10.0f), 10.0f)); }

template <class V, class S>
__device__ __forceinline__ V splat(S x) {
  return V{x, x, x, x};
}

template <class V, class S>
__device__ __forceinline__ V load4(const S* p) {
  return *reinterpret_cast<const V*>(p);
}

// Four f32 biases as chain accumulators (rounded to f16 in that profile).
template <class A4>
__device__ __forceinline__ A4 bias4(const float* p) {
  const float4 b = *reinterpret_cast<const float4*>(p);
  typedef decltype(A4{}[0]) E;
  return A4{(E)b.x, (E)b.y, (E)b.z, (E)b.w};
}

// Whether a kernel behind resident launches leaves window b as it is.
__device__ __forceinline__ bool decoded_before(const TdtArgs& a, uint32_t b) {
  return a.aborted && (a.aborted[2 * (b / a.aborted_windows) * kTdtSyncStride] == 0u ||
                       (a.after_team && !(a.status[b] & kTdtSyncTimeout)));
}

// Exchanged values: relaxed agent-scope atomics, coherent between XCDs.
__device__ __forceinline__ float xload(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void xstore(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t xload(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void xstore(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace
}  // namespace pk

#endif
