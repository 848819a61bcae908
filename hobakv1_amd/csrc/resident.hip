// The resident PCG: one launch runs up to `iters` whole iterations of each instance's (inner) solve
// with the instance's matrix held on the chip.
//
// The two-kernel iteration of solver_kernels.hip reads the matrix once per iteration and pays two
// launches for it: 28 us an iteration for a 79 MB FP64 matrix (40^3 lattice), about 11 us for a
// few hundred vertices, where nothing but the launches and their dependent loads is left.  The chip's
// registers and LDS hold 168 MB, so here an instance's rows are dealt out to W workgroups of one
// compute unit each, every workgroup loads its slots once, and an iteration moves only the
// vector entries its rows couple to.
//
// Arithmetic.  Every sum runs in the order of the two-kernel iteration: a row's blocks by the lane that
// handles them there, p.t by SpMV workgroup (four slices), r.r and r.z by update workgroup (four
// chunks of 21 R rows), and the totals over those partial sums by the same 256-lane tree.  The results
// are therefore bitwise those of the two-kernel iteration, whatever W is, and a solve may pass from
// one to the other at any even iteration.
//
// Work split.  Workgroup w owns a contiguous range of update workgroups' rows [ua, ub) and computes the
// slices that cover it, plus the rest of the SpMV workgroups (of four slices) that begin in it; the
// few rows past the range are computed twice, which costs less than handing t across workgroups.
//   registers  the first kReg 64-slot steps of each wave (9 values and a 16-bit place per slot);
//   LDS        the vector entries the slots couple to (FP64: p, which every workgroup keeps up to date
//              itself from z; FP32: z), t, and as many further steps as fit; the steps past that
//              are read from memory each iteration.
//
// Exchange.  Two all-to-all waits per iteration: on the p.t partial sums, and on the r.r / r.z partial
// sums, which also order z.  A partial sum is published as two 8-byte words that carry half of its
// bits and the iteration's tag each, so the wait and the read are one load, there is nothing to
// reset, and no address sees more than one writer.  Two copies alternate: a workgroup writes a copy
// again only after every workgroup has published the step in between, hence has read it.  z and the
// words are stored and loaded with agent-scope (L2-coherent) accesses; z's stores are
// waited for before the partial sums that announce them.  All other data is private to a workgroup or
// constant for the launch, so no cache is written back or invalidated: with a release and an acquire
// the same wait costs about 10 us more over 256 workgroups.  Measured alone: 2.6 us for both waits over 8
// workgroups, 6.6 us over 256.
//
// Residency.  An instance's workgroups wait for each other, so all of them must run at once.
// Workgroups take tickets, and tickets are dealt to instances in order, so at most the last instance
// whose workgroups have begun is incomplete and every other one makes progress.  Before a workgroup
// changes anything it announces itself and waits for the others of its instance; if they do not appear in
// time (another program holds the compute units) or one of them cannot hold its columns, the
// instance is left untouched and counted in Ctl::res_abort, and the host runs the two-kernel form.
#include "kernels.h"
#include "pcg_device.h"

namespace hobak {

namespace {

typedef unsigned long long u64;
constexpr int kResThreads = 512;
constexpr int kResWaves = kResThreads / 64;
constexpr int kResLds = 160 * 1024 - 1024;    // dynamic; the rest holds the static arrays below
constexpr int kAbort = 1 << 30;
constexpr u64 kJoinTicks = 20000000ull;       // 0.2 s of the 100 MHz wall clock
constexpr u64 kWaitTicks = 500000000ull;      // 5 s; every peer is running, so this is never reached

// 64-slot steps of a wave held in registers: 162 registers of values and 5 or 9 of places, which
// leaves about 80 of the 256 a wave may use at two waves per SIMD.
template <typename T>
constexpr int kReg = sizeof(T) == 8 ? 8 : 16;

__device__ __forceinline__ u64 ld_word(const HOBAK_GLOBAL u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_word(HOBAK_GLOBAL u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A vector entry that other workgroups write or read in this launch (all: through the caches, when
// the instance has one workgroup).
__device__ __forceinline__ double ld_shared(const HOBAK_GLOBAL double* p, bool all) {
  return all ? *p : __longlong_as_double((long long)ld_word((const HOBAK_GLOBAL u64*)p));
}
__device__ __forceinline__ float ld_shared(const HOBAK_GLOBAL float* p, bool all) {
  return all ? *p
             : __uint_as_float(__hip_atomic_load((const HOBAK_GLOBAL unsigned*)p, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void st_shared(HOBAK_GLOBAL double* p, double v, bool all) {
  if (all)
    *p = v;
  else
    st_word((HOBAK_GLOBAL u64*)p, (u64)__double_as_longlong(v));
}
__device__ __forceinline__ void st_shared(HOBAK_GLOBAL float* p, float v, bool all) {
  if (all)
    *p = v;
  else
    __hip_atomic_store((HOBAK_GLOBAL unsigned*)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void publish_word(HOBAK_GLOBAL u64* s, double v, unsigned tag) {
  const u64 b = (u64)__double_as_longlong(v);
  st_word(s, (b & 0xffffffffull) | ((u64)tag << 32));
  st_word(s + 1, (b >> 32) | ((u64)tag << 32));
}

// This lane's share (i0, i0 + 256, ...) of n published partial sums, added in ascending order; up to
// five are in flight at once.
__device__ __forceinline__ double poll_parts(const HOBAK_GLOBAL u64* s, int n, int i0, unsigned tag, int* failed) {
  constexpr int KP = 5;
  double v = 0.0;
  for (int base = i0; base < n; base += 256 * KP) {
    u64 lo[KP], hi[KP];
    u64 t0 = 0;
    for (int spin = 0;; spin++) {
      bool ready = true;
#pragma unroll
      for (int k = 0; k < KP; k++) {
        const int i = base + 256 * k < n ? base + 256 * k : base;
        lo[k] = ld_word(s + 2 * (size_t)i);
        hi[k] = ld_word(s + 2 * (size_t)i + 1);
      }
#pragma unroll
      for (int k = 0; k < KP; k++) ready = ready && (unsigned)(lo[k] >> 32) == tag && (unsigned)(hi[k] >> 32) == tag;
      if (ready) break;
      if ((spin & 255) == 255) {
        const u64 now = wall_clock64();
        if (t0 == 0) t0 = now;
        if (now - t0 > kWaitTicks) {
          *failed = 1;
          return 0.0;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < KP; k++)
      if (base + 256 * k < n) v += __longlong_as_double((long long)((lo[k] & 0xffffffffull) | (hi[k] << 32)));
  }
  return v;
}

// A load at a 32-bit byte offset from a uniform base (hobak_check_offsets keeps instances in range).
template <typename P>
__device__ __forceinline__ P ld_off(const HOBAK_GLOBAL P* base, unsigned byte_off) {
  return *(const HOBAK_GLOBAL P*)((const HOBAK_GLOBAL char*)base + byte_off);
}
template <typename P>
__device__ __forceinline__ HOBAK_GLOBAL P* at_off(HOBAK_GLOBAL P* base, unsigned byte_off) {
  return (HOBAK_GLOBAL P*)((HOBAK_GLOBAL char*)base + byte_off);
}

// A pointer field of the record, as a global pointer in scalar registers.  The record is read after the
// ticket's atomic, so the compiler does not use scalar loads by itself, and two dozen fields
// would each take vector registers that the matrix needs.
template <typename P>
__device__ __forceinline__ HOBAK_GLOBAL P* uptr(P* p) {
  const u64 b = (u64)p;
  const unsigned lo = (unsigned)uniform_i((int)(unsigned)b), hi = (unsigned)uniform_i((int)(unsigned)(b >> 32));
  return (HOBAK_GLOBAL P*)(((u64)hi << 32) | lo);
}

__device__ __forceinline__ int al16(int x) { return (x + 15) & ~15; }

template <typename T, int R>
__device__ __forceinline__ void resident_solve(const HOBAK_GLOBAL InstDev* __restrict__ I, int lb, int W,
                                               int iters, char* lds) {
  constexpr bool kF32 = sizeof(T) < sizeof(double);
  constexpr int NR = kReg<T>;
  constexpr int UR = 84 * R;                  // rows of an update workgroup
  constexpr int kStepBytes = 64 * 9 * (int)sizeof(T);
  __shared__ double red[2][5][4];             // wave sums of the two reductions
  __shared__ int scan[kResWaves], rest_of[kResWaves];
  __shared__ int sh_flag, sh_failed;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto ctl = ctl_of(I);
  const auto S = &ctl->sc[0];
  if (S->done) return;
  const int nrows = uniform_i(I->nv);
  const size_t ns = (size_t)uniform_i(I->nslots);
  const int sh = uniform_i(I->shift), H = 1 << sh;
  const int NU = uniform_i(I->nb[K_UPD]), NQ = uniform_i(I->nb[K_SPMV]);
  const auto slice_off = uptr(I->slice_off);
  const auto col = uptr(I->col);
  const auto A = uptr((const T*)I->A);
  const auto mi = uptr((const T*)I->minv);
  const auto ainv = uptr((const T*)I->agg_inv);
  const auto pinned = uptr(I->pinned);
  auto xg = uptr((T*)I->x);
  auto rg = uptr((T*)I->r);
  auto zg = uptr((T*)I->z);
  auto p0 = uptr((T*)I->p0);
  auto tg = uptr((T*)I->t);
  auto words = uptr(I->xwords);
  const auto prr = uptr(I->part_rr), prz = uptr(I->part_rz), pug = uptr(I->part_upd_g);
  const int precond = uniform_i(I->precond);
  const bool coarse = kF32 && uniform_i(I->coarse) != 0;
  const bool local = kF32 && uniform_i(I->agg) != 0;
  const int nval = coarse ? 5 : 2;
  bool first = uniform_i(S->first) != 0;
  double absNew = uniform_f(S->absNew), beta_d = uniform_f(S->beta), resNorm2 = uniform_f(S->resNorm2);
  int it_count = uniform_i(S->iters), status = uniform_i(S->status), done = 0;
  const double threshold = uniform_f(S->threshold);
  const int maxIters = uniform_i(S->maxIters);
  const unsigned epoch = (unsigned)uniform_i((int)ctl->res_epoch);
  double ce0 = 0.0, ce1 = 0.0, ce2 = 0.0, ai0 = 0.0, ai1 = 0.0, ai2 = 0.0;
  if (coarse) {
    ce0 = uniform_f(S->e[0]);
    ce1 = uniform_f(S->e[1]);
    ce2 = uniform_f(S->e[2]);
    ai0 = uniform_f(ctl->ac_inv[0]);
    ai1 = uniform_f(ctl->ac_inv[1]);
    ai2 = uniform_f(ctl->ac_inv[2]);
  }
  const bool solo = W == 1;
  // this workgroup's update workgroups, rows, SpMV workgroups and slices
  const int u0 = (int)((long)lb * NU / W), u1 = (int)((long)(lb + 1) * NU / W);
  const int nu = u1 - u0, nch = 4 * nu;
  const int ua = u0 * UR, ub = min(u1 * UR, nrows);
  const int nslices = (nrows + H - 1) >> sh;
  const int q0 = (ua + 4 * H - 1) >> (sh + 2), q1 = (ub + 4 * H - 1) >> (sh + 2);
  const int nq = q1 - q0;
  const int sa = ua >> sh;
  int sb = (ub + H - 1) >> sh;
  if (nq > 0) sb = max(sb, min(4 * q1, nslices));
  const int nsl = sb - sa;
  const int row0 = sa << sh;
  const int nrl = min(sb << sh, nrows) - row0;
  // the wave's slices sa + wave + 8 j: lane j holds the j-th one's first slot and step count
  const int nslw = nsl > wave ? (nsl - wave + kResWaves - 1) / kResWaves : 0;
  int l_beg = 0, l_nit = 0;
  if (lane < nslw) {
    const int s = sa + wave + kResWaves * lane;
    l_beg = slice_off[s];
    l_nit = (slice_off[s + 1] - l_beg) >> 6;
  }
  int steps = l_nit;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) steps += __shfl_xor(steps, off, 64);
  steps = __builtin_amdgcn_readfirstlane(steps);
  const int nrest = steps > NR ? steps - NR : 0;
  // LDS layout, first part (sizes known from the ranges)
  int off = 0;
  double* ptsl = (double*)(lds + off);  // p.t of each slice
  off += 8 * nsl;
  double* uw = (double*)(lds + off);    // sums of each chunk
  off += 8 * 5 * nch;
  double* lp = (double*)(lds + off);    // solo: the partial sums
  off += 8 * (nq + 5 * nu);
  off = al16(off);
  T* Tv = (T*)(lds + off);              // t (FP32: t_old between iterations)
  off += (int)sizeof(T) * 3 * nrl;
  T *Pv = nullptr, *Sv = Tv, *Dv = nullptr;
  if (kF32) {
    Pv = (T*)(lds + off);               // p of the own rows
    Sv = Pv + 3 * nrl;                  // the rows' sums before the diagonal term and t_old
    Dv = Sv + 3 * nrl;                  // the difference form's diagonal
    off += (int)sizeof(T) * 9 * nrl;
  }
  off = al16(off);
  const int nw = (nrows + 31) >> 5;     // the column set as a bitmap, at the top while it is built
  const int bm_off = kResLds - 2 * al16(4 * nw);
  unsigned* bm = (unsigned*)(lds + bm_off);
  unsigned* pre = (unsigned*)(lds + bm_off + al16(4 * nw));
  if (lane == 0) rest_of[wave] = nrest;
  if (tid == 0) sh_failed = 0;
  bool fits = nslw <= 64 && off <= bm_off;
  fits = __syncthreads_and(fits);
  int NC = 0, rest_base = 0, rest_all = 0;
  for (int w = 0; w < kResWaves; w++) {
    if (w < wave) rest_base += rest_of[w];
    rest_all += rest_of[w];
  }
  int* clist = (int*)(lds + off);
  T* zp = nullptr;
  unsigned short* idxr = nullptr;
  if (fits) {
    for (int i = tid; i < nw; i += kResThreads) bm[i] = 0u;
    __syncthreads();
    for (int i = tid; i < nrl; i += kResThreads) atomicOr(&bm[(row0 + i) >> 5], 1u << ((row0 + i) & 31));
    const int send = slice_off[sb];
    for (int i = slice_off[sa] + tid; i < send; i += kResThreads) {
      const int c = col[i];
      atomicOr(&bm[c >> 5], 1u << (c & 31));
    }
    __syncthreads();
    const int per = (nw + kResThreads - 1) / kResThreads;
    const int wa = min(tid * per, nw), wb = min(wa + per, nw);
    int cnt = 0;
    for (int i = wa; i < wb; i++) cnt += __popc(bm[i]);
    int inc = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane == 63) scan[wave] = inc;
    __syncthreads();
    int run = inc - cnt;
    for (int w = 0; w < kResWaves; w++) {
      if (w < wave) run += scan[w];
      NC += scan[w];
    }
    // second part: the column list, the vector entries, the places of the steps not in registers
    off += al16(4 * NC);
    zp = (T*)(lds + off);
    off += al16((kF32 ? 16 : 24) * NC);
    idxr = (unsigned short*)(lds + off);
    off += 128 * rest_all;
    fits = NC < 65536 && off <= bm_off;
    if (fits)
      for (int i = wa; i < wb; i++) {
        pre[i] = run;
        for (unsigned m = bm[i]; m; m &= m - 1) clist[run++] = 32 * i + __ffs(m) - 1;
      }
    __syncthreads();
  }
  // announce this workgroup (or that its instance cannot run here)
  auto arr = (HOBAK_GLOBAL int*)&ctl->res_arrive;
  if (tid == 0) {
    if (fits)
      __hip_atomic_fetch_add(arr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      __hip_atomic_fetch_or(arr, kAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (fits) {
    auto rank = [&](int c) -> int { return pre[c >> 5] + __popc(bm[c >> 5] & ((1u << (c & 31)) - 1u)); };
    const int own0 = rank(row0);
    // the register steps and their places; a step past the wave's last one multiplies zeros
    T m[NR][9];
    unsigned ix[(NR + 1) / 2];
    u64 ends = 0;  // bit k: step k (of the register steps) is the last one of its slice
    int cj = 0, cs = 0;  // cursor: the wave's slice and the step in it
    auto skip_empty = [&](int& js) {
      while (js < nslw && __builtin_amdgcn_readlane(l_nit, js) == 0) js++;
    };
    skip_empty(cj);
#pragma unroll
    for (int k = 0; k < NR; k++) {
      int id = 0;
#pragma unroll
      for (int e = 0; e < 9; e++) m[k][e] = T(0);
      if (k < steps) {
        const unsigned slot = (unsigned)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
        id = rank(ld_off(col, 4u * slot));
#pragma unroll
        for (int e = 0; e < 9; e++) m[k][e] = ld_off(A + e * ns, (unsigned)sizeof(T) * slot);
        if (++cs == __builtin_amdgcn_readlane(l_nit, cj)) {
          ends |= 1ull << k;
          cs = 0;
          cj++;
          skip_empty(cj);
        }
      }
      if (k & 1)
        ix[k >> 1] |= (unsigned)id << 16;
      else
        ix[k >> 1] = (unsigned)id;
    }
    const int rest_cj = cj, rest_cs = cs;  // where the steps past the registers begin
    for (int k = 0; k < nrest; k++) {
      const size_t slot = (size_t)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
      idxr[64 * (rest_base + k) + lane] = (unsigned short)rank(col[slot]);
      if (++cs == __builtin_amdgcn_readlane(l_nit, cj)) {
        cs = 0;
        cj++;
        skip_empty(cj);
      }
    }
    __syncthreads();  // the bitmap is not read past here: its space goes to the LDS steps
    off = al16(off);
    const int share = (kResLds - off) / kStepBytes / kResWaves;  // LDS steps of each wave
    const int nlds = min(nrest, share);
    T* ml = (T*)(lds + off) + (size_t)wave * share * (64 * 9);
    cj = rest_cj;
    cs = rest_cs;
    for (int k = 0; k < nlds; k++) {
      const size_t slot = (size_t)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
#pragma unroll
      for (int e = 0; e < 9; e++) ml[(9 * k + e) * 64 + lane] = A[e * ns + slot];
      if (++cs == __builtin_amdgcn_readlane(l_nit, cj)) {
        cs = 0;
        cj++;
        skip_empty(cj);
      }
    }
    for (int i = tid; i < 3 * nrl; i += kResThreads) {
      const size_t g = 3 * (size_t)row0 + i;
      if (kF32) {
        Tv[i] = first ? T(0) : tg[g];
        Pv[i] = first ? T(0) : p0[g];
        Sv[i] = T(0);
        Dv[i] = (T)gbl(I->dg)[g];
      } else {
        Tv[i] = T(0);
      }
    }
    if (!kF32 && !first)
      for (int i = tid; i < NC; i += kResThreads) {
        const size_t g = 3 * (size_t)clist[i];
#pragma unroll
        for (int c = 0; c < 3; c++) zp[3 * i + c] = p0[g + c];
      }
    // wait for the instance's other workgroups
    if (tid == 0) {
      const u64 t0 = wall_clock64();
      int v = __hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      while (!(v & kAbort) && v < W) {
        if (wall_clock64() - t0 > kJoinTicks)
          __hip_atomic_compare_exchange_strong(arr, &v, v | kAbort, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
        else
          __builtin_amdgcn_s_sleep(1);
        v = __hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      sh_flag = (v & kAbort) ? 0 : 1;
    }
    __syncthreads();
    if (sh_flag) {
      const int half = tid >> 8, i0 = tid & 255;
      const int tid_ = tid, lane_ = lane;
      const auto wpt = words;                          // p.t: [copy][NQ]
      const auto wup = words + 4 * (size_t)NQ;         // update sums: [copy][5][NU]
      int it = 0;
      for (; it < iters; it++) {
        const unsigned tag = epoch + 1u + (unsigned)it;  // this iteration's words
        // opaque copies: row numbers and addresses are formed anew in each iteration instead of being
        // kept in registers that the matrix needs
        int tid = tid_, lane = lane_;
        asm volatile("" : "+v"(tid), "+v"(lane));
        // finish the previous iteration: |r|^2, r.z (and the coarse correction's sums of r)
        double beta = 0.0;
        if (!first) {
          for (int k0 = 0; k0 < nval; k0 += 2) {
            const int kind = k0 + half;
            double v = 0.0;
            if (kind < nval) {
              if (it == 0) {  // left by the launch before
                const auto src = kind == 0 ? prr : kind == 1 ? prz : pug + (size_t)(kind - 2) * NU;
                for (int i = i0; i < NU; i += 256) v += src[i];
              } else if (solo) {
                for (int i = i0; i < NU; i += 256) v += lp[nq + kind * nu + i];
              } else if (i0 < NU) {
                v = poll_parts(wup + 2 * (size_t)(5 * ((tag - 1u) & 1u) + kind) * NU, NU, i0, tag - 1u, &sh_failed);
              }
            }
            v = wave_sum(v);
            if (lane == 0 && kind < nval) red[0][kind][wave & 3] = v;
          }
          __syncthreads();
          if (sh_failed) {
            done = 1;
            status = 2;
            break;
          }
          double tot[5];
#pragma unroll
          for (int k = 0; k < 5; k++) {
            tot[k] = 0.0;
            if (k < nval)
#pragma unroll
              for (int w = 0; w < 4; w++) tot[k] += red[0][k][w];
            tot[k] = uniform_f(tot[k]);
          }
          const double rrv = tot[0];
          double rz = tot[1];
          if (coarse) {
            ce0 = ai0 * tot[2];
            ce1 = ai1 * tot[3];
            ce2 = ai2 * tot[4];
            rz += tot[2] * ce0 + tot[3] * ce1 + tot[4] * ce2;
          }
          resNorm2 = rrv;
          if (nonfinite(rrv) || !(rz == rz)) {
            done = 1;
            status = 2;
            break;
          }
          if (rrv < threshold) {
            done = 1;
            break;
          }
          beta = rz / absNew;
          beta = uniform_f(beta);
          beta_d = beta;
          absNew = rz;
          it_count++;
          if (it_count >= maxIters) {
            done = 1;
            status = 1;
            break;
          }
        }
        const T bt = (T)beta;
        // the vector entries the slots couple to: z, or (FP64) p = z + beta p_old
        for (int b0 = tid; b0 < NC; b0 += 4 * kResThreads) {
          int cc[4];
          T zv[4][3];
#pragma unroll
          for (int j = 0; j < 4; j++) cc[j] = clist[min(b0 + j * kResThreads, NC - 1)];
#pragma unroll
          for (int j = 0; j < 4; j++)
#pragma unroll
            for (int c = 0; c < 3; c++) zv[j][c] = ld_shared(at_off(zg + c, 3u * (unsigned)sizeof(T) * (unsigned)cc[j]), solo);
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const int i = b0 + j * kResThreads;
            if (i >= NC) continue;
            if (kF32) {
              *(float4*)(zp + 4 * i) = make_float4((float)zv[j][0], (float)zv[j][1], (float)zv[j][2], 0.f);
            } else {
#pragma unroll
              for (int c = 0; c < 3; c++) zp[3 * i + c] = first ? zv[j][c] : fma(bt, zp[3 * i + c], zv[j][c]);
            }
          }
        }
        __syncthreads();
        // A times those entries, slice by slice
        {
          int js = 0;
          T s0 = T(0), s1 = T(0), s2 = T(0), d0 = T(0), d1 = T(0), d2 = T(0);
          auto own_entry = [&]() {  // FP32: the row's own z, which its columns are relative to
            if (!kF32 || js >= nslw) return;
            const int r = ((sa + wave + kResWaves * js) << sh) + (lane & (H - 1));
            const bool live = r < nrows;
            const T* o = zp + 4 * (own0 + (live ? r : row0) - row0);
            d0 = live ? o[0] : T(0);
            d1 = live ? o[1] : T(0);
            d2 = live ? o[2] : T(0);
          };
          auto gather = [&](int id, T(&v)[3]) {
            if (kF32) {
              const float4 q = *(const float4*)(zp + 4 * id);
              v[0] = (T)q.x;
              v[1] = (T)q.y;
              v[2] = (T)q.z;
            } else {
              v[0] = zp[3 * id];
              v[1] = zp[3 * id + 1];
              v[2] = zp[3 * id + 2];
            }
          };
          auto accumulate = [&](const T(&a)[9], const T(&v)[3]) {
            const T p0v = kF32 ? v[0] - d0 : v[0], p1v = kF32 ? v[1] - d1 : v[1], p2v = kF32 ? v[2] - d2 : v[2];
            s0 = row3(s0, a[0], a[1], a[2], p0v, p1v, p2v);
            s1 = row3(s1, a[3], a[4], a[5], p0v, p1v, p2v);
            s2 = row3(s2, a[6], a[7], a[8], p0v, p1v, p2v);
          };
          auto finish_slice = [&]() {
            if (H == 8) {
              s0 += map32(s0, [](unsigned b) { return dpp<kRor8>(b); });
              s1 += map32(s1, [](unsigned b) { return dpp<kRor8>(b); });
              s2 += map32(s2, [](unsigned b) { return dpp<kRor8>(b); });
            }
            if (H <= 16) {
              s0 = add_xor16(s0);
              s1 = add_xor16(s1);
              s2 = add_xor16(s2);
            }
            if (H <= 32) {
              s0 = add_xor32(s0);
              s1 = add_xor32(s1);
              s2 = add_xor32(s2);
            }
            const int rl = ((wave + kResWaves * js) << sh) + lane;
            if (lane < H && rl < nrl) {
              Sv[3 * rl] = s0;
              Sv[3 * rl + 1] = s1;
              Sv[3 * rl + 2] = s2;
            }
            s0 = s1 = s2 = T(0);
            js++;
            skip_empty(js);
            own_entry();
          };
          skip_empty(js);
          own_entry();
          // the register steps in groups whose gathers are issued together (those past the wave's
          // last step multiply zeros)
          constexpr int G = kF32 ? 4 : 2;
#pragma unroll
          for (int k0 = 0; k0 < NR; k0 += G) {
            if (k0 < steps) {
              T v[G][3];
#pragma unroll
              for (int k = k0; k < k0 + G && k < NR; k++)
                gather((int)((k & 1) ? ix[k >> 1] >> 16 : ix[k >> 1] & 0xffffu), v[k - k0]);
#pragma unroll
              for (int k = k0; k < k0 + G && k < NR; k++) {
                accumulate(m[k], v[k - k0]);
                if ((ends >> k) & 1) finish_slice();
              }
            }
          }
          int kj = rest_cj, ks = rest_cs;
          for (int k = 0; k < nrest; k++) {
            T a[9];
            if (k < nlds) {
#pragma unroll
              for (int e = 0; e < 9; e++) a[e] = ml[(9 * k + e) * 64 + lane];
            } else {
              const unsigned slot = (unsigned)(__builtin_amdgcn_readlane(l_beg, kj) + 64 * ks + lane);
#pragma unroll
              for (int e = 0; e < 9; e++) a[e] = ld_off(A + e * ns, (unsigned)sizeof(T) * slot);
            }
            T v[3];
            gather((int)idxr[64 * (rest_base + k) + lane], v);
            accumulate(a, v);
            if (++ks == __builtin_amdgcn_readlane(l_nit, kj)) {
              ks = 0;
              kj++;
              skip_empty(kj);
              finish_slice();
            }
          }
        }
        // t and p of the rows, and p.t of each slice
        for (int j = 0; j < nslw; j++) {
          const int ls = wave + kResWaves * j;
          const int rl = (ls << sh) + lane;
          double pt = 0.0;
          if (lane < H && rl < nrl) {
            T s0 = Sv[3 * rl], s1 = Sv[3 * rl + 1], s2 = Sv[3 * rl + 2];
            if (kF32) {
              const T* o = zp + 4 * (own0 + rl);
              T z0 = o[0], z1 = o[1], z2 = o[2];
              if (coarse) {
                z0 += (T)ce0;
                z1 += (T)ce1;
                z2 += (T)ce2;
              }
              s0 = fma(Dv[3 * rl], z0, s0);
              s1 = fma(Dv[3 * rl + 1], z1, s1);
              s2 = fma(Dv[3 * rl + 2], z2, s2);
              if (!first) {
                s0 = fma(bt, Tv[3 * rl], s0);
                s1 = fma(bt, Tv[3 * rl + 1], s1);
                s2 = fma(bt, Tv[3 * rl + 2], s2);
                z0 = fma(bt, Pv[3 * rl], z0);
                z1 = fma(bt, Pv[3 * rl + 1], z1);
                z2 = fma(bt, Pv[3 * rl + 2], z2);
              }
              Tv[3 * rl] = s0;
              Tv[3 * rl + 1] = s1;
              Tv[3 * rl + 2] = s2;
              Pv[3 * rl] = z0;
              Pv[3 * rl + 1] = z1;
              Pv[3 * rl + 2] = z2;
              pt = dot3((double)z0, (double)z1, (double)z2, (double)s0, (double)s1, (double)s2);
            } else {
              const T* o = zp + 3 * (own0 + rl);
              pt = dot3((double)o[0], (double)o[1], (double)o[2], (double)s0, (double)s1, (double)s2);
            }
          }
          pt = wave_sum(pt);
          if (lane == 0) ptsl[ls] = pt;
        }
        __syncthreads();
        if (tid < nq) {
          double s = 0.0;
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const int sl = 4 * (q0 + tid) + w;
            s += sl < nslices ? ptsl[sl - sa] : 0.0;
          }
          if (solo)
            lp[tid] = s;
          else
            publish_word(wpt + 2 * ((size_t)(tag & 1u) * NQ + q0 + tid), s, tag);
        }
        if (solo) __syncthreads();
        // alpha, then x, r and z of the own rows, chunk by chunk; the first chunk's loads are issued
        // before the wait for p.t
        const int c = lane - 3 * (lane / 3);
        const int bse = lane - c;
        T rv0[R], xv[R], m0[R], m1[R], m2[R];
        unsigned char pn[R];
        auto load = [&](int cl) {
#pragma unroll
          for (int q = 0; q < R; q++) {
            const int row = ((4 * u0 + cl) * R + q) * 21 + lane / 3;
            rv0[q] = xv[q] = m0[q] = m1[q] = m2[q] = T(0);
            pn[q] = 1;
            if (lane < 63 && row < nrows) {
              const unsigned i = (unsigned)(3 * row + c);
              if (local) pn[q] = ld_off(pinned, (unsigned)row);
              constexpr unsigned ts = sizeof(T);
              rv0[q] = ld_off(rg, ts * i);
              xv[q] = ld_off(xg, ts * i);
              if (precond == 0) {
                m0[q] = ld_off(mi, ts * i);
              } else {
                m0[q] = ld_off(mi, 3 * ts * i);
                m1[q] = ld_off(mi + 1, 3 * ts * i);
                m2[q] = ld_off(mi + 2, 3 * ts * i);
              }
            }
          }
        };
        if (wave < nch) load(wave);
        if (half == 0) {
          double v = 0.0;
          if (solo) {
            for (int i = i0; i < NQ; i += 256) v += lp[i];
          } else if (i0 < NQ) {
            v = poll_parts(wpt + 2 * (size_t)(tag & 1u) * NQ, NQ, i0, tag, &sh_failed);
          }
          v = wave_sum(v);
          if (lane == 0) red[1][0][wave] = v;
        }
        __syncthreads();
        if (sh_failed) {
          done = 1;
          status = 2;
          break;
        }
        double ptt = 0.0;
#pragma unroll
        for (int w = 0; w < 4; w++) ptt += red[1][0][w];
        const T alpha = (T)(absNew / uniform_f(ptt));
        for (int cl = wave; cl < nch; cl += kResWaves) {
          if (cl != wave) load(cl);
          T rq[R], zq[R];
          double rr2 = 0.0, rz = 0.0, gc = 0.0;
#pragma unroll
          for (int q = 0; q < R; q++) {
            const int row = ((4 * u0 + cl) * R + q) * 21 + lane / 3;
            const bool live = lane < 63 && row < nrows;
            const unsigned i = (unsigned)(3 * row + c);
            T rv = T(0);
            if (live) {
              const int rl = row - row0;
              const T pv = kF32 ? Pv[3 * rl + c] : zp[3 * (own0 + rl) + c];
              *at_off(xg, (unsigned)sizeof(T) * i) = fma(alpha, pv, xv[q]);
              rv = fma(-alpha, Tv[3 * rl + c], rv0[q]);
              *at_off(rg, (unsigned)sizeof(T) * i) = rv;
            }
            const T r0 = __shfl(rv, bse, 64);
            const T r1 = __shfl(rv, bse + 1, 64);
            const T r2 = __shfl(rv, bse + 2, 64);
            rq[q] = rv;
            zq[q] = precond == 0 ? m0[q] * rv : fma(m2[q], r2, fma(m0[q], r0, m1[q] * r1));
          }
          if constexpr (kF32) {
            if (local) agg_correct<T, R>(ainv, 4 * u0 + cl < (nrows + 21 * R - 1) / (21 * R) ? 4 * u0 + cl : 0,
                                         c, rq, pn, zq);
          }
#pragma unroll
          for (int q = 0; q < R; q++) {
            const int row = ((4 * u0 + cl) * R + q) * 21 + lane / 3;
            if (lane < 63 && row < nrows) {
              st_shared(at_off(zg, (unsigned)sizeof(T) * (unsigned)(3 * row + c)), zq[q], solo);
              rr2 = fma((double)rq[q], (double)rq[q], rr2);
              rz = fma((double)rq[q], (double)zq[q], rz);
              gc += (double)rq[q];
            }
          }
          const double v0 = wave_sum(rr2), v1 = wave_sum(rz);
          if (lane == 0) {
            uw[cl] = v0;
            uw[nch + cl] = v1;
          }
          if (coarse) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
              const double g = wave_sum(c == k ? gc : 0.0);
              if (lane == 0) uw[(2 + k) * nch + cl] = g;
            }
          }
        }
        // z is complete before the sums that announce it are published
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid < nval * nu) {
          const int kind = tid / nu, u = tid - kind * nu;
          double s = 0.0;
#pragma unroll
          for (int w = 0; w < 4; w++) s += uw[kind * nch + 4 * u + w];
          if (solo)
            lp[nq + kind * nu + u] = s;
          else
            publish_word(wup + 2 * ((size_t)(5 * (tag & 1u) + kind) * NU + u0 + u), s, tag);
          if (it == iters - 1) {  // the next launch finishes this iteration from these
            auto dst = kind == 0 ? prr : kind == 1 ? prz : pug + (size_t)(kind - 2) * NU;
            dst[u0 + u] = s;
          }
        }
        if (solo) __syncthreads();
        first = false;
      }
      __syncthreads();
      if (!done)  // the solve goes on in another launch: its p and t
        for (int i = tid; i < 3 * (ub - ua); i += kResThreads) {
          const size_t g = 3 * (size_t)ua + i;
          const int l = 3 * (ua - row0) + i;
          p0[g] = kF32 ? Pv[l] : zp[3 * own0 + l];
          if (kF32) tg[g] = Tv[l];
        }
      if (lb == 0 && tid == 0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
          auto N = &ctl->sc[k];
          if (k == 1) {
            N->rhsNorm2 = S->rhsNorm2;
            N->threshold = threshold;
            N->alpha = S->alpha;
            N->maxR = S->maxR;
            N->maxIters = maxIters;
          }
          N->absNew = absNew;
          N->beta = beta_d;
          N->resNorm2 = resNorm2;
          N->iters = it_count;
          N->done = done;
          N->status = status;
          N->first = first ? 1 : 0;
        }
        ctl->spmv_work += (unsigned)it;
        ctl->res_epoch = epoch + 2u + (unsigned)it;
      }
    }
  }
  // the last workgroup to leave clears the instance's meeting point
  __syncthreads();
  if (tid == 0) {
    auto ex = (HOBAK_GLOBAL int*)&ctl->res_exit;
    if (__hip_atomic_fetch_add(ex, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == W - 1) {
      if (__hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kAbort) ctl->res_abort += 1;
      __hip_atomic_store(arr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(ex, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// b: boff[i] counts the workgroups of instance i.  tickets: [0] the next ticket, [1] workgroups done;
// both zero between launches.
template <typename T, int R>
__global__ __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void cg_resident_kernel(
    Batch b, int* tickets, int iters) {
  extern __shared__ __align__(16) char lds[];
  __shared__ int sh_ticket;
  if (threadIdx.x == 0)
    sh_ticket = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  int lb, W;
  const HOBAK_GLOBAL InstDev* I = seg_find(b, __builtin_amdgcn_readfirstlane(sh_ticket), lb, W);
  resident_solve<T, R>(I, lb, W, iters, lds);
  if (threadIdx.x == 0 &&
      __hip_atomic_fetch_add(tickets + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == b.total - 1) {
    __hip_atomic_store(tickets, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(tickets + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <typename T, int R>
hipError_t resident_r(const Batch& b, int* tickets, int iters, hipStream_t s) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&cg_resident_kernel<T, R>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kResLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((cg_resident_kernel<T, R>), dim3(b.total), dim3(kResThreads), kResLds, s, b, tickets, iters);
  return hipGetLastError();
}

}  // namespace

size_t resident_words(int nb_spmv, int nb_upd) { return 4 * (size_t)nb_spmv + 20 * (size_t)nb_upd; }

template <typename T>
hipError_t launch_cg_resident(const Batch& b, int groups, int* tickets, int iters, hipStream_t s) {
  if (b.total <= 0) return hipSuccess;
  switch (groups) {
    case 1: return resident_r<T, 1>(b, tickets, iters, s);
    case 2: return resident_r<T, 2>(b, tickets, iters, s);
    case 4: return resident_r<T, 4>(b, tickets, iters, s);
    default: return hipErrorInvalidValue;
  }
}
template hipError_t launch_cg_resident<double>(const Batch&, int, int*, int, hipStream_t);
template hipError_t launch_cg_resident<float>(const Batch&, int, int*, int, hipStream_t);

}  // namespace hobak
