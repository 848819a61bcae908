// Device helpers shared by the PCG kernels of solver_kernels.hip and resident.hip, which must agree
// bitwise.
#pragma once
#include <cfloat>

#include "kernels.h"

namespace hobak {

// v of lane i ^ 32 and i ^ 16 (the swap exchanges halves, or odd and even rows, of two registers; with one
// value in both, each lane finds its partner's in one of the two results), and of lane i ^ 8.
__device__ __forceinline__ unsigned xor32(unsigned v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return (threadIdx.x & 32) ? r[0] : r[1];
}
__device__ __forceinline__ unsigned xor16(unsigned v) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return (threadIdx.x & 16) ? r[0] : r[1];
}
template <int CTRL>
__device__ __forceinline__ unsigned dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int kRor8 = 0x128, kRor4 = 0x124, kQuad2301 = 0x4e, kQuad1032 = 0xb1;

template <typename F>
__device__ __forceinline__ float map32(float v, F&& f) {
  return __uint_as_float(f(__float_as_uint(v)));
}
template <typename F>
__device__ __forceinline__ double map32(double v, F&& f) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return __longlong_as_double((long long)((unsigned long long)f((unsigned)(b >> 32)) << 32 | f((unsigned)b)));
}
// v + v of lane i ^ 32, and + v of lane i ^ 16.
template <typename T>
__device__ __forceinline__ T add_xor32(T v) {
  return v + map32(v, [](unsigned b) { return xor32(b); });
}
template <typename T>
__device__ __forceinline__ T add_xor16(T v) {
  return v + map32(v, [](unsigned b) { return xor16(b); });
}
// Sum over the wave, in every lane: a butterfly over lanes i ^ 32, 16, 8, 4, 2, 1.  Each step adds the
// same two values in both lanes, so every lane ends with the same bits, and after the i ^ 8 step a
// row of 16 repeats with period 8, so a rotation by 4 reads lane i ^ 4.  The moves are register-file
// ones (swaps and DPP); as six ds_bpermute steps the sum took about 0.3 us, and several stand in a
// PCG iteration's serial chain.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  v = add_xor32(v);
  v = add_xor16(v);
  v += map32(v, [](unsigned b) { return dpp<kRor8>(b); });
  v += map32(v, [](unsigned b) { return dpp<kRor4>(b); });
  v += map32(v, [](unsigned b) { return dpp<kQuad2301>(b); });
  v += map32(v, [](unsigned b) { return dpp<kQuad1032>(b); });
  return v;
}

// A value that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ int uniform_i(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform_f(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform_f(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// s + (m0 p0 + m1 p1 + m2 p2) with its two fused multiply-adds spelled out.  Kernels that must
// agree bitwise (the SpMV's variants, the FP64 two-kernel and p-form iterations) then contract
// the products the same way, whatever the compiler would pick for each.
template <typename T>
__device__ __forceinline__ T row3(T s, T m0, T m1, T m2, T p0, T p1, T p2) {
  return s + fma(m2, p2, fma(m0, p0, m1 * p1));
}
// a0 b0 + a1 b1 + a2 b2 in FP64 with its fused multiply-adds spelled out (for the same reason).
__device__ __forceinline__ double dot3(double a0, double a1, double a2, double b0, double b1, double b2) {
  return fma(a2, b2, fma(a1, b1, a0 * b0));
}

__device__ __forceinline__ bool nonfinite(double v) { return !(v == v) || v > DBL_MAX || v < -DBL_MAX; }

// Local aggregate correction of update chunk ch (rows (ch * R + q) * 21 + lane / 3, component
// c = lane % 3 of each, as in the update kernel): g = P_I^T r over the chunk's free rows, summed
// in a fixed lane order to the same value in every lane, then z += (P_I^T A P_I)^-1 g at the free
// rows.  pn[q] != 0: row q is pinned or past the end.  Every lane of the wave takes part.
template <typename T, int R>
__device__ __forceinline__ void agg_correct(const HOBAK_GLOBAL T* ainv, int ch, int c, const T (&rq)[R],
                                            const unsigned char (&pn)[R], T (&zq)[R]) {
  T s = T(0);
#pragma unroll
  for (int q = 0; q < R; q++) s += pn[q] ? T(0) : rq[q];
  const T g0 = wave_sum(c == 0 ? s : T(0));
  const T g1 = wave_sum(c == 1 ? s : T(0));
  const T g2 = wave_sum(c == 2 ? s : T(0));
  const HOBAK_GLOBAL T* m = ainv + 9 * (size_t)ch + 3 * c;
  const T e = fma(m[2], g2, fma(m[1], g1, m[0] * g0));
#pragma unroll
  for (int q = 0; q < R; q++)
    if (!pn[q]) zq[q] += e;
}

}  // namespace hobak
