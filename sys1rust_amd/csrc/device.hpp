// Device-side helpers shared by the HIP kernels of libsys1hip (gfx950 / CDNA4 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace s1 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// bf16 values travel as raw uint16_t in memory.
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// f32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32; NaN stays NaN).
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }

// Two f32 -> two bf16 in one register (low half = a), one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  bf16x2 r;
  r[0] = static_cast<__bf16>(a);
  r[1] = static_cast<__bf16>(b);
  return __builtin_bit_cast(uint32_t, r);
}

// The 16-bit element type of weights and activations, a template parameter of every kernel that
// touches them: bf16 (the default) or f16 (the checkpoints' own type, setting dtype=f16). Both
// feed the 32x32x16 MFMA at the same rate; the traits give the MFMA opcode and the conversions
// (f32 -> 16 bit rounds to nearest even, v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
struct Bf16 {
  typedef __bf16 scalar;
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float f32(uint16_t h) { return bf2f(h); }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) { return s1::pack2(a, b); }
  static __device__ __forceinline__ uint16_t bits(float f) { return f2bf(f); }
};
// f32 -> f16 rounds the f32 value as computed. Without the opaque copy the compiler may fuse the
// conversion into the FMA that produced the value (v_fma_mix*_f16: one rounding, straight to
// f16), so two kernels that compute the same f32 value could store f16 values that differ in the
// last bit, depending on which of them it fused. (bf16 has no such fused form.)
struct F16 {
  typedef _Float16 scalar;
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 v2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float f32(uint16_t h) { return float(__builtin_bit_cast(_Float16, h)); }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    asm("" : "+v"(a), "+v"(b));
    v2 r;
    r[0] = static_cast<_Float16>(a);
    r[1] = static_cast<_Float16>(b);
    return __builtin_bit_cast(uint32_t, r);
  }
  static __device__ __forceinline__ uint16_t bits(float f) {
    asm("" : "+v"(f));
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
  }
};

// A split f32 value: hi + lo / 2048, two f16 (hi the value rounded, lo what that leaves, scaled up so
// that it keeps its bits below the smallest hi): 23 significant bits, one less than f32. Three
// quarters of the f32 values are held exactly and the others to 2^-23 (4.2e-8 in the root mean
// square over a binade), for values down to 2^-28 of f16's largest; weights that come from f16 or
// bf16 are exact. (The split and its scaling by 2^11: Ootomo and Yokota, "Recovering single
// precision accuracy from Tensor Cores while surpassing the FP32 theoretical peak performance",
// 2022.) Operands of the f32 products are held so, times a power of two that keeps them in range; a row keeps its bytes, [32 hi | 32 lo] for every 32 elements: element e of a
// matrix (rows a multiple of 32) has hi at 16-bit index split_at(e) and lo 32 after it.
__host__ __device__ inline size_t split_at(size_t e) { return (e & ~size_t(31)) * 2 + (e & 31); }
template <int N>  // N consecutive values (a multiple of 2), scaled by sc
__device__ __forceinline__ void split_f16(const float* v, float sc, uint32_t* hi, uint32_t* lo) {
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    float x[2], r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) x[e] = v[2 * i + e] * sc;
    hi[i] = F16::pack2(x[0], x[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) r[e] = (x[e] - F16::f32(uint16_t(e ? hi[i] >> 16 : hi[i]))) * 2048.0f;
    lo[i] = F16::pack2(r[0], r[1]);
  }
}
// Four values at element e (a multiple of 4) of a split matrix.
__device__ __forceinline__ void store4_split(void* m, size_t e, const float* v, float sc) {
  uint32_t hi[2], lo[2];
  split_f16<4>(v, sc, hi, lo);
  uint16_t* o = static_cast<uint16_t*>(m) + split_at(e);
  *reinterpret_cast<uint2*>(o) = make_uint2(hi[0], hi[1]);
  *reinterpret_cast<uint2*>(o + 32) = make_uint2(lo[0], lo[1]);
}

// Between LDS writes and reads of what other lanes of the same wave wrote: a wave's LDS accesses take
// effect in order, so this only keeps the compiler, which knows one lane's accesses, from reordering them.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 8 elements of type E held in a uint4 <-> floats.
template <class E>
__device__ __forceinline__ void unpack8(const uint4& v, float* f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = E::f32(uint16_t(w[i]));
    f[2 * i + 1] = E::f32(uint16_t(w[i] >> 16));
  }
}
template <class E>
__device__ __forceinline__ uint4 pack8(const float* f) {
  return make_uint4(E::pack2(f[0], f[1]), E::pack2(f[2], f[3]), E::pack2(f[4], f[5]), E::pack2(f[6], f[7]));
}

// The first `valid` (0..8) 16-bit elements of an 8-element piece, the rest zeroed, by selects.
__device__ __forceinline__ uint4 keep_first(uint4 v, int valid) {
  auto m = [valid](int e) { return (valid > e ? 0x0000ffffu : 0u) | (valid > e + 1 ? 0xffff0000u : 0u); };
  v.x &= m(0);
  v.y &= m(2);
  v.z &= m(4);
  v.w &= m(6);
  return v;
}

// Cross-lane steps on the VALU: DPP moves within a row of 16 lanes (quad_perm for lane ^ 1 and
// lane ^ 2, row_half_mirror and row_mirror to join 4- and 8-lane groups), and gfx950's
// v_permlane16_swap / v_permlane32_swap between rows and between the wave's halves. A
// __shfl_xor is a ds_bpermute through the LDS pipe: a reduction of 6 of them in a chain waits on
// 6 LDS round trips.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// x and the value of lane l ^ 16 (within each half), as a pair (own row's first).
__device__ __forceinline__ void swap16(float v, float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// The value of lane l % 32 and of lane l % 32 + 32, in every lane.
__device__ __forceinline__ void swap32(float v, float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// v(l) + v(l ^ 32) and max(v(l), v(l ^ 32)), the same bits in both lanes.
__device__ __forceinline__ float half_sum(float v) {
  float a, b;
  swap32(v, a, b);
  return a + b;
}
__device__ __forceinline__ float half_max(float v) {
  float a, b;
  swap32(v, a, b);
  return fmaxf(a, b);
}

// Sum / max over the 64 lanes of a wavefront; every lane gets the same bits (each step combines
// the same two partial results in the same order in every lane).
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<0xb1>(v);   // quad_perm(1, 0, 3, 2): lane ^ 1
  v += dpp<0x4e>(v);   // quad_perm(2, 3, 0, 1): lane ^ 2
  v += dpp<0x141>(v);  // row_half_mirror: the other quad of the 8
  v += dpp<0x140>(v);  // row_mirror: the other 8 of the 16
  float a, b;
  swap16(v, a, b);
  return half_sum(a + b);
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp<0xb1>(v));
  v = fmaxf(v, dpp<0x4e>(v));
  v = fmaxf(v, dpp<0x141>(v));
  v = fmaxf(v, dpp<0x140>(v));
  float a, b;
  swap16(v, a, b);
  return half_max(fmaxf(a, b));
}

// GELU with the error function, 0.5 x (1 + erf(x / sqrt 2)), erf by Abramowitz & Stegun 7.1.26:
// for z = |x| / sqrt 2 and t = 1 / (1 + p z), 1 - erf(z) = (a1 t + ... + a5 t^5) exp(-z^2) with
// |error| <= 1.5e-7. For x < 0, 1 + erf(x / sqrt 2) is that tail itself (no cancellation). In f32
// the GELU is within 4.2e-7 absolute of the exact one on [-12, 12], and within 1.7e-4 relative
// wherever |GELU| > 1e-3: a tenth of a bf16 ulp at most. It costs one reciprocal, one exp2 and
// five FMAs, a third of the library erff with its range branches.
__device__ __forceinline__ float gelu_erf(float x) {
  const float z = fabsf(x) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, z, 1.0f));
  float poly = fmaf(1.061405429f, t, -1.453152027f);
  poly = fmaf(poly, t, 1.421413741f);
  poly = fmaf(poly, t, -0.284496736f);
  poly = fmaf(poly, t, 0.254829592f);
  const float q = poly * t * __builtin_amdgcn_exp2f(-(z * z) * 1.4426950408889634f);  // 1 - erf(z)
  return 0.5f * x * (x >= 0.0f ? 2.0f - q : q);
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD b % 8). Remap the
// hardware block index so that consecutive logical tiles sit on one XCD and share its L2.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int x = b & 7, i = b >> 3;
  return x * q + (x < r ? x : r) + i;
}

}  // namespace s1
