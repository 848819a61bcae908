// Device helpers shared by the PCG kernels of solver_kernels.hip and resident.hip, which must agree
// bitwise.
#pragma once
#include <cfloat>

#include "kernels.h"

namespace hobak {

// (a, b) with a's upper 32 lanes and b's lower 32 exchanged (SWAP32), or a's odd rows of 16 lanes and b's even
// ones (SWAP16).  a + b then holds, in each half (or each row of a pair), the sum over lanes i and i ^ 32
// (i ^ 16) of what was a and of what was b: one addition reduces two values, and with a == b every
// lane ends with its own sum.
enum { SWAP32, SWAP16 };
template <int W>
__device__ __forceinline__ void lane_swap(unsigned& a, unsigned& b) {
  const auto r = W == SWAP32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false)
                             : __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
template <int W>
__device__ __forceinline__ float swap_add(float x, float y) {
  unsigned a = __float_as_uint(x), b = __float_as_uint(y);
  lane_swap<W>(a, b);
  return __uint_as_float(a) + __uint_as_float(b);
}
template <int W>
__device__ __forceinline__ double swap_add(double x, double y) {
  const unsigned long long xb = (unsigned long long)__double_as_longlong(x);
  const unsigned long long yb = (unsigned long long)__double_as_longlong(y);
  unsigned al = (unsigned)xb, ah = (unsigned)(xb >> 32), bl = (unsigned)yb, bh = (unsigned)(yb >> 32);
  lane_swap<W>(al, bl);
  lane_swap<W>(ah, bh);
  return __longlong_as_double((long long)((unsigned long long)ah << 32 | al)) +
         __longlong_as_double((long long)((unsigned long long)bh << 32 | bl));
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
// Sum over each row of 16 lanes, in every lane: a butterfly over lanes i ^ 8, 4, 2, 1.  After the i ^ 8 step
// a row repeats with period 8, so a rotation by 4 reads lane i ^ 4.
template <typename T>
__device__ __forceinline__ T row_sum(T v) {
  v += map32(v, [](unsigned b) { return dpp<kRor8>(b); });
  v += map32(v, [](unsigned b) { return dpp<kRor4>(b); });
  v += map32(v, [](unsigned b) { return dpp<kQuad2301>(b); });
  v += map32(v, [](unsigned b) { return dpp<kQuad1032>(b); });
  return v;
}
// Sum over the wave, in every lane: a butterfly over lanes i ^ 32, 16, 8, 4, 2, 1.  Each step adds the
// same two values in both lanes, so every lane ends with the same bits.  The moves are register-file ones
// (swaps and DPP); as six ds_bpermute steps the sum took about 0.3 us, and several stand in a PCG
// iteration's serial chain.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  v = swap_add<SWAP32>(v, v);
  v = swap_add<SWAP16>(v, v);
  return row_sum(v);
}
// wave_sum of a in lanes 0-31 and of b in lanes 32-63, for about the price of one.
__device__ __forceinline__ double wave_sum2(double a, double b) {
  double v = swap_add<SWAP32>(a, b);
  v = swap_add<SWAP16>(v, v);
  return row_sum(v);
}
// wave_sum of each group of H consecutive lanes, in each of its lanes (the other lanes' zeros left out, which
// change nothing).
template <int H>
__device__ __forceinline__ double group_sum(double v) {
  if (H == 64) v = swap_add<SWAP32>(v, v);
  if (H >= 32) v = swap_add<SWAP16>(v, v);
  return row_sum(v);
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
__device__ __forceinline__ void agg_apply(const T (&m)[3], int c, const T (&rq)[R], const unsigned char (&pn)[R],
                                          T (&zq)[R]) {
  T s = T(0);
#pragma unroll
  for (int q = 0; q < R; q++) s += pn[q] ? T(0) : rq[q];
  const T g0 = wave_sum(c == 0 ? s : T(0));
  const T g1 = wave_sum(c == 1 ? s : T(0));
  const T g2 = wave_sum(c == 2 ? s : T(0));
  const T e = fma(m[2], g2, fma(m[1], g1, m[0] * g0));
#pragma unroll
  for (int q = 0; q < R; q++)
    if (!pn[q]) zq[q] += e;
}
template <typename T, int R>
__device__ __forceinline__ void agg_correct(const HOBAK_GLOBAL T* ainv, int ch, int c, const T (&rq)[R],
                                            const unsigned char (&pn)[R], T (&zq)[R]) {
  const HOBAK_GLOBAL T* p = ainv + 9 * (size_t)ch + 3 * c;
  const T m[3] = {p[0], p[1], p[2]};
  agg_apply<T, R>(m, c, rq, pn, zq);
}

}  // namespace hobak
