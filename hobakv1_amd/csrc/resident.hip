// The resident PCG: one launch runs up to `iters` whole iterations of each instance's (inner) solve
// with the instance's matrix held on the chip.
//
// The two-kernel iteration of solver_kernels.hip reads the matrix once per iteration and pays two
// launches for it: 28 us an iteration for a 79 MB FP64 matrix (40^3 lattice), about 11 us for a
// few hundred vertices, where nothing but the launches and their dependent loads is left.  The chip's
// registers and LDS hold 168 MB, so here an instance's rows are dealt out to W workgroups of one
// compute unit each, every workgroup loads its slots once, and an iteration moves only the
// vector entries its rows couple to.  Measured per iteration: 10.4 us for the 40^3 lattice (FP64, 206
// workgroups; FP32 9.4), 5.2 us for 10^3 (8 workgroups of one die), 4.0 us for 4^3 (one).
//
// Arithmetic (all but BIG).  Every sum runs in the order of the two-kernel iteration: a row's blocks by the lane that
// handles them there, p.t by SpMV workgroup (four slices), r.r and r.z by update workgroup (four
// chunks of 21 R rows), and the totals over those partial sums by the same 256-lane tree.  The results
// are therefore bitwise those of the two-kernel iteration, whatever W is, and a solve may pass from
// one to the other at any even iteration.
//
// Work split.  Workgroup w owns a contiguous range of update workgroups' rows [ua, ub) and computes the
// slices that cover it, plus, past kSplitMax and with 16-row slices, the rest of the SpMV workgroups (of four
// slices) that begin in it; the few rows past the range are computed twice, which costs less than handing t
// across workgroups.
//   registers  the first kReg 64-slot steps of each wave (9 values and a 16-bit place per slot);
//   LDS        the vector entries the slots couple to (FP64: p, which every workgroup keeps up to date
//              itself from z; FP32: z), t, and as many further steps as fit, dealt so that the
//              waves stream equally; the steps past that are read from memory each iteration.
//
// BIG is the reduced-precision form for more rows than the update workgroups cover in one run each (86,016
// with two row groups), where the two-kernel form is bound by reading 160 MB of matrix and 30 MB of vectors an
// iteration: 46 us for 303,242 vertices.  It runs on every compute unit, which hold about half the
// matrix and stream the rest: 29 us, of which 13 for the product (90 MB streamed, 7 TB/s) and 5 for the update's
// vectors.  Its rows are dealt in single chunks of 21 R, and each workgroup publishes one word per sum; the
// sums are so added in another order than the two-kernel form's (the same in every launch).  They
// are FP64 sums behind FP32 step lengths, which that has not changed in any run.  FP64 solves keep the
// two-kernel form there: their results depend on the order to 1e-8 (one iteration more or less at the end),
// and the update workgroups' runs of rows lie too far apart for one workgroup's columns.
//
// What bounds it.  With the matrix on chip an iteration is two waits plus a serial chain in which every
// wave of a SIMD issues a few hundred instructions, so the loop is written for few instructions: places
// are LDS byte offsets, a slice's three sums are reduced by swapping lanes between them, both dot
// products share one lane reduction, rows past the end are handled by the buffer descriptors'
// bounds, and addresses are formed anew instead of being kept where they would push the matrix out of
// its registers.  That took the 40^3 FP64 iteration from 15.7 us to 10.6.
//
// Exchange.  Two all-to-all waits per iteration: on the p.t partial sums, and on the r.r / r.z partial
// sums, which also order z.  A partial sum is published as one 16-byte word that carries its bits in two
// halves next to the iteration's tag, so the wait and the read are one load, there is nothing to
// reset, and no address sees more than one writer.  Two copies alternate: a workgroup writes a copy
// again only after every workgroup has published the step in between, hence has read it; likewise z is
// overwritten only after every workgroup has published its p.t (or a zero), hence has read z.  While four
// waves collect r.r and r.z, the other four wait for the few workgroups whose z this one needs and read it.
// z and the words are stored and loaded device-coherently, past the dies' L2s; z's stores are
// waited for before the partial sums that announce them.  All other data is private to a workgroup or
// constant for the launch, so no cache is written back or invalidated: with a release and an acquire
// the same wait costs about 10 us more over 256 workgroups.  One wait measured alone: 1.4 us over 8
// workgroups, 2.5 us over 206 with 539 to 1077 words (3.2 us with 8-byte loads and 8-byte words; 2.3 us
// with eight copies of each word or a second level of sums, which was not worth their code).
//
// One die.  Up to eight instances of at most 32 workgroups each are placed on one die (XCD) each, where z and the
// words go to the die's own L2 by ordinary stores: both waits then take about 1000 cycles less of an
// iteration's 13,000 (10^3 FP64 step 783 -> 686 us, 17x9x23 BDF 2.37 -> 2.03 ms).  The loads are the same, past the
// compute unit's cache (a load of workgroup scope may be served from that cache and never see the
// word).  Workgroups learn their die from the hardware and take its tickets; an instance whose die gets too few
// workgroups is left untouched.
//
// Residency.  An instance's workgroups wait for each other, so all of them must run at once.
// Workgroups take tickets, and tickets are dealt to instances in order, so at most the last instance
// whose workgroups have begun is incomplete and every other one makes progress.  Before a workgroup
// changes anything it announces itself and waits for the others of its instance; if they do not appear in
// time (another program holds the compute units) or one of them cannot hold its columns, the
// instance is left untouched and counted in Ctl::res_abort, and in Ctl::res_late where only time ran out: the
// host then takes another form for good, or for a while.  Workgroups that have met run until the launch ends, so the
// waits of its iterations are short; but where several processes share the device, their queues take turns, and two
// launches that each got only part of their compute units back wait in vain (the likely cause; with four processes
// waits were in vain once in some 10,000 launches).  A workgroup that waits too long marks the instance
// (Ctl::res_lost) and leaves, as all others then do; the host starts that solve again from its right-hand side.
#include "kernels.h"
#include "pcg_device.h"

#include <algorithm>

namespace hobak {

namespace {

typedef unsigned long long u64;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr int kResThreads = 512;
constexpr int kResWaves = kResThreads / 64;
constexpr int kResLds = 160 * 1024 - 2048;    // dynamic; the rest holds the static arrays below
constexpr int kResMaxUpd = 512;               // update workgroups of an instance
// Up to this many SpMV workgroups (of four slices), a workgroup publishes p.t only of the slices that begin in
// its rows: the sum of those that follow a group's first one, and each of the others of a group that begins in
// another workgroup's rows by itself, so that the four are still added in order.  Without that it computes
// the rest of its last group's rows a second time, up to 255 rows past its own 168 to 336 with 64-row slices.  A
// lane then polls up to four words, so the rule ends where lanes would have more than one group each.
constexpr int kSplitMax = 255;
constexpr int kMisfit = 1 << 30, kLate = kResLate, kAbort = kMisfit | kLate, kLost = kResLost;  // of Ctl::res_arrive
// How long an instance's workgroups wait for each other, in ticks of the 100 MHz wall clock: they are dispatched
// together, so they meet within microseconds unless other work holds compute units: earlier instances of the
// same launch, or another process's launch, which ends within milliseconds to tens of them, or whose workgroups wait
// in vain too because this launch holds the compute units they lack.  On every compute unit, 20 ms, so that of such
// two the other goes on (with 0.2 s for all, four processes that step 303,242, 68,921, 9,261 and 1,331 vertices took
// 0.2 to 0.8 s for a step now and then); otherwise 50 ms; on one die, of which a large instance of another
// process may leave too few compute units although others are free, 1 ms, after which the instance rather runs over the
// whole device.
template <bool BIG, bool ONE>
constexpr u64 kJoinTicks = ONE ? 100000ull : BIG ? 2000000ull : 5000000ull;
constexpr unsigned kWaitTicks = 10000000u;    // 0.1 s: the longest wait in an iteration (see Residency above)
constexpr int kAgentScope = 16;               // cache policy of a buffer access: coherent over the device's L2s
constexpr int kDieScope = 0;                  // of a store: to this die's L2, where loads of the other policy find it
constexpr int kArrived = 1023;                // Ctl::res_arrive: workgroups here

// 64-slot steps of a wave held in registers: 162 or 144 registers of values and 5 or 8 of places, of the
// 256 a wave may use at two waves per SIMD.
template <typename T>
constexpr int kReg = sizeof(T) == 8 ? 9 : 16;
// Streamed steps whose values are on their way at once: every workgroup of the BIG form streams about half its
// steps (72x61x66 step: 19.4 ms with one a wave under way, 19.0 with two).
template <bool BIG>
constexpr int kAhead = BIG ? 2 : 1;

typedef __amdgpu_buffer_rsrc_t Rsrc;
// A buffer descriptor of `bytes` bytes: accesses past them read zero and write nothing.
__device__ __forceinline__ Rsrc buffer(void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00027000);
}
template <typename T, int AUX = 0>
__device__ __forceinline__ T buf_ld(Rsrc rs, unsigned off, int soff = 0) {
  if constexpr (sizeof(T) == 8) {
    const u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(rs, off, soff, AUX);
    return __longlong_as_double((long long)((u64)q.y << 32 | q.x));
  } else {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, soff, AUX));
  }
}
template <int AUX>
__device__ __forceinline__ void buf_st(Rsrc rs, unsigned off, double v) {
  const u64 b = (u64)__double_as_longlong(v);
  const u32x2 q = {(unsigned)b, (unsigned)(b >> 32)};
  __builtin_amdgcn_raw_buffer_store_b64(q, rs, off, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void buf_st(Rsrc rs, unsigned off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, off, 0, AUX);
}
// The three entries of a vertex that another workgroup wrote in this launch.
__device__ __forceinline__ void ld_vertex(Rsrc rs, unsigned off, double (&v)[3]) {
  const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, kAgentScope);
  const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 16, 0, kAgentScope);
  v[0] = __longlong_as_double((long long)((u64)q.y << 32 | q.x));
  v[1] = __longlong_as_double((long long)((u64)q.w << 32 | q.z));
  v[2] = __longlong_as_double((long long)((u64)w.y << 32 | w.x));
}
__device__ __forceinline__ void ld_vertex(Rsrc rs, unsigned off, float (&v)[3]) {
  const u32x3 q = __builtin_amdgcn_raw_buffer_load_b96(rs, off, 0, kAgentScope);
  v[0] = __uint_as_float(q.x);
  v[1] = __uint_as_float(q.y);
  v[2] = __uint_as_float(q.z);
}

// A published value: its low and high word, each next to the tag of its iteration (8-byte halves are
// stored and loaded whole, so both tags match only where both words are this iteration's).
template <int SC>
__device__ __forceinline__ void publish_word(Rsrc rs, unsigned i, double v, unsigned tag) {
  const u64 b = (u64)__double_as_longlong(v);
  const u32x4 q = {(unsigned)b, tag, (unsigned)(b >> 32), tag};
  __builtin_amdgcn_raw_buffer_store_b128(q, rs, 16u * i, 0, SC);
}

// Spins until the K published values at byte offsets o[k] carry `tag`; gives up (false) after kWaitTicks.
// All of a round's loads are in flight together.
template <int K>
__device__ __forceinline__ bool poll_words(Rsrc rs, const unsigned (&o)[K], unsigned tag, double (&v)[K]) {
  u32x4 q[K];
  unsigned t0 = 0;
  for (int spin = 0;; spin++) {
    asm volatile("" ::: "memory");  // each round loads anew
#pragma unroll
    for (int k = 0; k < K; k++) q[k] = __builtin_amdgcn_raw_buffer_load_b128(rs, o[k], 0, kAgentScope);
    unsigned miss = 0;
#pragma unroll
    for (int k = 0; k < K; k++) miss |= (q[k].y ^ tag) | (q[k].w ^ tag);
    if (miss == 0) break;
    if ((spin & 255) == 255) {
      const unsigned now = (unsigned)wall_clock64() | 1u;
      if (t0 == 0) t0 = now;
      if (now - t0 > kWaitTicks) return false;
    }
  }
#pragma unroll
  for (int k = 0; k < K; k++) v[k] = __longlong_as_double((long long)((u64)q[k].z << 32 | q[k].x));
  return true;
}

// This lane's share (i0, i0 + 256, ...) of each of NK runs of n published values, KP of a run in flight at once,
// added in ascending order; run k begins at byte base + k * 16 n.
template <int NK, int KP>
__device__ __forceinline__ void poll_parts(Rsrc rs, unsigned base, int n, int i0, unsigned tag, int* failed,
                                           double (&sum)[NK]) {
#pragma unroll
  for (int k = 0; k < NK; k++) sum[k] = 0.0;
  for (int b = i0; b < n; b += 256 * KP) {
    unsigned o[NK * KP];
    double v[NK * KP];
#pragma unroll
    for (int j = 0; j < KP; j++) {
      o[j] = base + 16u * (unsigned)(j == 0 || b + 256 * j < n ? b + 256 * j : b);
#pragma unroll
      for (int k = 1; k < NK; k++) o[KP * k + j] = o[j] + 16u * (unsigned)(k * n);
    }
    if (!poll_words<NK * KP>(rs, o, tag, v)) {
      *failed = 1;
      return;
    }
#pragma unroll
    for (int k = 0; k < NK; k++)
#pragma unroll
      for (int j = 0; j < KP; j++)
        if (j == 0 || b + 256 * j < n) sum[k] += v[KP * k + j];
  }
}
template <int NK>
__device__ __forceinline__ void poll_sums(Rsrc rs, unsigned base, int n, int i0, unsigned tag, int* failed,
                                          double (&sum)[NK]) {
  if (n <= 256)
    poll_parts<NK, 1>(rs, base, n, i0, tag, failed, sum);
  else if (NK > 1 || n <= 512)
    poll_parts<NK, 2>(rs, base, n, i0, tag, failed, sum);
  else
    poll_parts<NK, 5>(rs, base, n, i0, tag, failed, sum);
}

// A load at a 32-bit byte offset from a uniform base (hobak_check_offsets keeps instances in range).
template <typename P>
__device__ __forceinline__ P ld_off(const HOBAK_GLOBAL P* base, unsigned byte_off) {
  return *(const HOBAK_GLOBAL P*)((const HOBAK_GLOBAL char*)base + byte_off);
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

// nonfinite() from the exponent bits alone (no constants held in registers).
__device__ __forceinline__ bool not_finite(double v) {
  return ((unsigned)((u64)__double_as_longlong(v) >> 52) & 0x7ffu) == 0x7ffu;
}

// The die (XCD, with an L2 of its own) this wave runs on: HW_REG_XCC_ID, bits 0 to 3.
__device__ __forceinline__ int die_of_wave() { return __builtin_amdgcn_s_getreg(20 | 3 << 11) & 7; }

__device__ __forceinline__ int al16(int x) { return (x + 15) & ~15; }

template <typename T, int R, int H, bool BIG, bool ONE>
__device__ __forceinline__ void resident_solve(const HOBAK_GLOBAL InstDev* __restrict__ I, int lb, int W,
                                               int iters, char* lds) {
  constexpr bool kF32 = sizeof(T) < sizeof(double);
  constexpr int NR = kReg<T>, ND = kAhead<BIG>;
  constexpr unsigned ts = sizeof(T);
  constexpr int SC = ONE ? kDieScope : kAgentScope;  // the exchange between workgroups
  constexpr int sh = H == 64 ? 6 : H == 32 ? 5 : 4, L = 64 / H;
  constexpr int UC = BIG ? 1 : 4;             // 21 R-row chunks of a unit of rows
  constexpr int UR = 21 * R * UC;             // its rows: an update workgroup's, or one chunk's
  constexpr int ZS = kF32 ? 16 : 24;          // bytes of a vertex in the LDS vector
  constexpr int GF = 4;                       // other workgroups' columns a thread has in flight at once
  constexpr int kStepBytes = 64 * 9 * (int)ts;
  __shared__ double red[2][5][4];             // wave sums of the two reductions
  __shared__ int scan[kResWaves], rest_of[kResWaves];
  __shared__ int sh_flag, sh_failed;
  __shared__ unsigned ubits[kResMaxUpd / 32];  // the update workgroups whose z this one reads, as bits ...
  __shared__ unsigned short need[kResMaxUpd];  // ... and as a list
  __shared__ unsigned char apart[256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto ctl = ctl_of(I);
  const auto S = &ctl->sc[0];
  if (S->done) return;
  const int nrows = uniform_i(I->nv);
  const size_t ns = (size_t)uniform_i(I->nslots);
  const int NB = uniform_i(I->nb[K_UPD]), NQ = uniform_i(I->nb[K_SPMV]);
  const int NU = BIG ? (nrows + UR - 1) / UR : NB;  // units of rows ...
  const int NX = BIG ? W : NU;                      // ... and words of each update sum
  const auto slice_off = uptr(I->slice_off);
  const auto col = uptr(I->col);
  const auto A = uptr((const T*)I->A);
  const auto ainv = uptr((const T*)I->agg_inv);
  const auto pinned = uptr(I->pinned);
  // fields that only a launch's first or last iteration needs are read where they are used: held through the
  // loop, they would not leave enough scalar registers
  auto rec = [&]() {
    auto J = I;
    asm volatile("" : "+s"(J));
    return J;
  };
  const int precond = uniform_i(I->precond);
  const unsigned vec_bytes = 3u * ts * (unsigned)nrows;
  const Rsrc rs_r = buffer((void*)uptr((T*)I->r), vec_bytes), rs_x = buffer((void*)uptr((T*)I->x), vec_bytes);
  const Rsrc rs_z = buffer((void*)uptr((T*)I->z), vec_bytes);
  const Rsrc rs_m = buffer((void*)uptr((T*)I->minv), (precond == 0 ? 1u : 3u) * vec_bytes);
  // whether p.t words are single slices' where a group of four straddles two workgroups (see kSplitMax)
  const bool split = !BIG && H >= 32 && W > 1 && NQ <= kSplitMax;
  const unsigned npt = BIG ? (unsigned)W : split ? 4u * (unsigned)(NQ + 1) : (unsigned)(NQ + NU);  // p.t words of a copy
  const Rsrc rs_w = buffer((void*)uptr(I->xwords), 32u * npt + 160u * (unsigned)NX);
  // (BIG: at most 64 steps of 512 x 256 threads, so the planes together stay below 2^30 bytes)
  const Rsrc rs_a = buffer((void*)uptr((T*)I->A), (unsigned)(9 * ns * ts));
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
  const bool solo = !BIG && W == 1;
  // this workgroup's units, rows, SpMV workgroups and slices
  // (as many units each, the last fewer: a 336-row workgroup then begins on a 16-row slice and has at most 24 of them,
  // three a wave; dealt evenly, most began half a slice off and the 25th slice of some, with the columns
  // past 1024 that it couples to, set the pace of all: 40^3 FP64 step 5.07 -> 4.85 ms.  BIG: NU W < 2^31, nv < 2^25)
  const int per = (NU + W - 1) / W;
  const int u0 = uniform_i(BIG ? lb * NU / W : min(lb * per, NU)), u1 = uniform_i(BIG ? (lb + 1) * NU / W : min((lb + 1) * per, NU));
  const int nu = u1 - u0, nch = UC * nu;
  const int ua = u0 * UR, ub = min(u1 * UR, nrows), nown = ub - ua;
  const int nslices = (nrows + H - 1) >> sh;
  auto first_q = [&](int row) { return (row + 4 * H - 1) >> (sh + 2); };  // the first SpMV workgroup from row on
  auto first_s = [&](int row) { return (row + H - 1) >> sh; };         // the first slice from row on
  const int q0 = first_q(ua), q1 = first_q(ub);
  const int nq = q1 - q0;
  // A workgroup in whose rows no SpMV workgroup (split: no slice) begins publishes a zero in its place, so
  // that nobody passes the wait on p.t, and overwrites z, before every workgroup has read it: np words in
  // all, this one's at qe
  const int ra = min(tid * per * UR, nrows), rb = min((tid + 1) * per * UR, nrows);
  const bool none = tid < W && (split ? first_s(ra) == first_s(rb) : first_q(ra) == first_q(rb));
  const int np = BIG ? W : NQ + __syncthreads_count(none), qe = BIG ? 0 : NQ + __syncthreads_count(none && tid < lb);
  const int sa = ua >> sh, so = first_s(ua);
  int sb = first_s(ub);
  const int nown_s = sb - so;  // the slices that begin in its rows
  if (!BIG && !split && nq > 0) sb = max(sb, min(4 * q1, nslices));
  if (tid < 256) {  // bits j: slice 4 tid + j is published by another workgroup than slice 4 tid
    auto owner = [&](int s) { return s * H / (UR * per); };
    unsigned m = 0;
    if (split && tid < NQ)
#pragma unroll
      for (int j = 1; j < 4; j++)
        if (4 * tid + j < nslices && owner(4 * tid + j) != owner(4 * tid)) m |= 1u << j;
    apart[tid] = (unsigned char)m;
  }
  const int nsl = sb - sa;
  const int row0 = sa << sh;
  const int nrl = min(sb << sh, nrows) - row0;
  const int nrp = nsl << sh;  // the rows of whole slices
  // the wave's slices sa + wave + 8 j: lane j holds the j-th one's first slot and step count (no slice is
  // empty: resident_pack)
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
  // the column set as a bitmap, at the bottom of the LDS, below what is written while it is needed
  const int nw = (nrows + 31) >> 5;
  const int bm_end = 2 * al16(4 * nw);
  unsigned* bm = (unsigned*)lds;
  unsigned* pre = (unsigned*)(lds + al16(4 * nw));
  if (lane == 0) rest_of[wave] = nrest;
  if (tid == 0) sh_failed = 0;
  bool fits = steps <= 64 && bm_end <= kResLds;
  fits = __syncthreads_and(fits);
  int NC = 0, rest_base = 0, rest_all = 0, nneed = 0;
  for (int w = 0; w < kResWaves; w++) {
    const int n = uniform_i(rest_of[w]);
    if (w < wave) rest_base += n;
    rest_all += n;
  }
  // LDS layout: vector entries, t (FP64: also the rows' z between update and next_p), FP32: p, the rows'
  // sums and the diagonal; partial sums; places of the steps not in registers; the column list; steps
  int off_t = 0, off_p = 0, off_s = 0, off_d = 0, off_pt = 0, off_u = 0, off_lp = 0, off_ix = 0, off_cl = 0, off_m = 0;
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
      const int n = uniform_i(scan[w]);
      if (w < wave) run += n;
      NC += n;
    }
    const int vec = 3 * (int)ts * nrp;
    off_t = al16(ZS * NC);
    off_s = off_t;
    off_p = off_t + vec;
    if (kF32) {
      off_s = off_p + vec;
      off_d = off_s + vec;
    }
    off_pt = al16(off_t + (kF32 ? 4 : 1) * vec);
    off_u = off_pt + 8 * nsl;
    off_lp = off_u + 8 * 5 * nch;
    off_ix = max(al16(off_lp + (solo ? 8 * (nq + 5 * nu) : split ? 2 * nsl : 0)), bm_end);
    off_cl = off_ix + 128 * rest_all;
    off_m = al16(off_cl + 4 * NC);
    fits = ZS * NC <= 65536 && off_m <= kResLds;
    if (fits)
      for (int i = wa; i < wb; i++) {
        pre[i] = run;
        for (unsigned m = bm[i]; m; m &= m - 1) ((int*)(lds + off_cl))[run++] = 32 * i + __ffs(m) - 1;
      }
    __syncthreads();
  }
  // announce this workgroup (or that its instance cannot run here)
  auto arr = (HOBAK_GLOBAL int*)&ctl->res_arrive;
  if (tid == 0) {
    if (fits)
      __hip_atomic_fetch_add(arr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      __hip_atomic_fetch_or(arr, kMisfit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (fits) {
    int* const clist = (int*)(lds + off_cl);
    T* const Tv = (T*)(lds + off_t);
    T* const Sv = (T*)(lds + off_s);
    T* const Pv = (T*)(lds + off_p);
    T* const Dv = (T*)(lds + off_d);
    double* const ptsl = (double*)(lds + off_pt);  // p.t of each slice
    double* const uw = (double*)(lds + off_u);     // sums of each chunk
    double* const lp = (double*)(lds + off_lp);    // solo: the partial sums
    // split: what to publish for each slice: the word, and in bits 12 to 14 how many slices it sums (5: a zero)
    unsigned short* const pubs = (unsigned short*)(lds + off_lp);
    unsigned short* const idxr = (unsigned short*)(lds + off_ix);
    auto rank = [&](int c) -> int { return pre[c >> 5] + __popc(bm[c >> 5] & ((1u << (c & 31)) - 1u)); };
    // the own rows' entries in the vector; the other workgroups' are [0, flo) and [flo + nown, NC)
    const int own0 = uniform_i(rank(row0)), flo = uniform_i(rank(ua)), nf = NC - nown;
    auto foreign = [&](int k) -> int { return k < flo ? k : k + nown; };
    for (int i = tid; i < kResMaxUpd / 32; i += kResThreads) ubits[i] = 0u;
    __syncthreads();
    for (int k = tid; k < nf; k += kResThreads) {
      int u = clist[foreign(k)] / UR;
      if (BIG) u = ((u + 1) * W - 1) / NU;  // the workgroup that owns the unit
      atomicOr(&ubits[u >> 5], 1u << (u & 31));
    }
    __syncthreads();
    for (int w = 0; w < (NX + 31) >> 5; w++) {
      const unsigned m = (unsigned)uniform_i((int)ubits[w]);
      if (tid >> 5 == w && (m >> (tid & 31) & 1u))
        need[nneed + __popc(m & ((1u << (tid & 31)) - 1u))] = (unsigned short)tid;
      nneed += __popc(m);
    }
    // the register steps and the places of their columns (byte offsets); a step past the wave's last one
    // multiplies zeros
    T m[NR][9];
    unsigned ix[(NR + 1) / 2];
    u64 ends = 0;  // bit k: step k is the last one of its slice
    int cj = 0, cs = 0;  // cursor: the wave's slice and the step in it
    auto advance = [&](int k) {
      if (++cs == __builtin_amdgcn_readlane(l_nit, cj)) {
        ends |= 1ull << k;
        cs = 0;
        cj++;
      }
    };
#pragma unroll
    for (int k = 0; k < NR; k++) {
      int id = 0;
#pragma unroll
      for (int e = 0; e < 9; e++) m[k][e] = T(0);
      if (k < steps) {
        const unsigned slot = (unsigned)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
        id = ZS * rank(ld_off(col, 4u * slot));
#pragma unroll
        for (int e = 0; e < 9; e++) m[k][e] = ld_off(A + e * ns, ts * slot);
        advance(k);
      }
      if (k & 1)
        ix[k >> 1] |= (unsigned)id << 16;
      else
        ix[k >> 1] = (unsigned)id;
    }
    const int rest_cj = cj, rest_cs = cs;  // where the steps past the registers begin
    for (int k = 0; k < nrest; k++) {
      const size_t slot = (size_t)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
      idxr[64 * (rest_base + k) + lane] = (unsigned short)(ZS * rank(col[slot]));
      advance(NR + k);
    }
    __syncthreads();  // the bitmap is not read past here: the vectors take its space
    if (split)
      for (int i = tid; i < nsl; i += kResThreads) {
        const int s = sa + i;
        unsigned e = 0;
        if (nown_s == 0)
          e = i == 0 ? 5u << 12 | 4u * (unsigned)qe : 0u;
        else if (s >= so && ((s & 3) == 0 || (s & ~3) < so))
          e = (unsigned)((s & 3) == 0 ? min(4, sb - s) : 1) << 12 | (unsigned)s;
        pubs[i] = (unsigned short)e;
      }
    // LDS steps of each wave: all but the last `streamed` of its steps past the registers, for the least
    // `streamed` that fits (the slowest wave of the slowest workgroup sets the pace)
    const int cap = (kResLds - off_m) / kStepBytes;
    int streamed = -1, taken = 0, before = 0;
    do {
      streamed++;
      taken = before = 0;
      for (int w = 0; w < kResWaves; w++) {
        const int n = max(uniform_i(rest_of[w]) - streamed, 0);
        if (w < wave) before += n;
        taken += n;
      }
    } while (taken > cap);
    const int nlds = uniform_i(max(nrest - streamed, 0));
    T* const ml = (T*)(lds + off_m) + (size_t)uniform_i(before) * (64 * 9);
    cj = rest_cj;
    cs = rest_cs;
    for (int k = 0; k < nlds; k++) {
      const size_t slot = (size_t)(__builtin_amdgcn_readlane(l_beg, cj) + 64 * cs + lane);
#pragma unroll
      for (int e = 0; e < 9; e++) ml[(9 * k + e) * 64 + lane] = A[e * ns + slot];
      advance(NR + k);
    }
    const int str_cj = cj, str_cs = cs;  // where the steps past the LDS begin
    // (z only ever by device-coherent loads here: an ordinary one would leave its line, with other workgroups'
    // rows, in this die's L2, where the coherent ones would then find it)
    const auto p0 = gbl((const T*)rec()->p0), tg = gbl((const T*)rec()->t);
    for (int i = tid; i < 3 * nrl; i += kResThreads) {
      const size_t g = 3 * (size_t)row0 + i;
      if (kF32) {
        Tv[i] = first ? T(0) : tg[g];
        Pv[i] = first ? T(0) : p0[g];
        Dv[i] = (T)gbl(I->dg)[g];
      } else {
        Tv[i] = buf_ld<T, kAgentScope>(rs_z, ts * (unsigned)g);
      }
    }
    if (kF32)
      for (int i = tid; i < 3 * nown; i += kResThreads)
        ((T*)lds)[4 * (flo + i / 3) + i % 3] = buf_ld<T, kAgentScope>(rs_z, ts * (unsigned)(3 * ua + i));
    else
      for (int i = tid; i < NC; i += kResThreads) {  // (in the first iteration beta is 0)
        const size_t g = 3 * (size_t)clist[i];
#pragma unroll
        for (int c = 0; c < 3; c++) ((T*)lds)[3 * i + c] = first ? T(0) : p0[g + c];
      }
    // wait for the instance's other workgroups
    if (tid == 0) {
      const u64 t0 = wall_clock64();
      int v = __hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      while (!(v & kAbort) && (v & kArrived) < W) {
        if (wall_clock64() - t0 > kJoinTicks<BIG, ONE>)
          __hip_atomic_compare_exchange_strong(arr, &v, v | kLate, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
        else
          __builtin_amdgcn_s_sleep(1);
        v = __hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      sh_flag = (v & kAbort) ? 0 : 1;
    }
    __syncthreads();
    if (sh_flag) {
      // words: p.t [copy][npt], then the update sums [copy][5][NU]
      const unsigned wup = 32u * npt, wstride = 80u * (unsigned)NX;
      // the update's rows of this lane: chunk `wave` of the workgroup, R rows 21 apart; the 64th lane has none
      int urow = lane < 63 ? (UC * u0 + wave) * 21 * R + lane / 3 : 0x7fffff;
      int c = lane - 3 * (lane / 3);
      unsigned gofs = lane < 63 ? ts * (unsigned)(3 * urow + c) : 0x7ffff000u;
      int srow = (wave << sh) + (lane & (H - 1));  // this lane's row in the wave's first slice
      int tid_ = tid;
      T* const zown = (T*)(lds + ZS * own0);
      int it = 0;
      // Where the loop's instructions lie against 32 bytes changes its time by 1% to 3%, and without this line every
      // change to the code before it moves them.  The best of the eight places, on one die: 24 bytes past a boundary (10^3
      // FP32 709 us, of 707 to 728; 17x9x23 FP64 1.983 ms, of 1.98 to 2.01); over the device: 4 in FP64 and 28 in
      // FP32 (40^3 step 4.83 ms, of 4.83 to 4.96, and 3.42, of 3.42 to 3.48).
      asm volatile(".p2align 8\n .rept %0\n s_nop 0\n .endr" ::"n"(ONE ? 6 : kF32 ? 7 : 1));
      for (; it < iters; it++) {
        const unsigned tag = epoch + 1u + (unsigned)it;  // this iteration's words
        const unsigned wprev = wup + ((tag - 1u) & 1u) * wstride;
        // opaque to the compiler: addresses derived from these are formed anew in each iteration
        // instead of being kept in registers that the matrix needs
        asm volatile("" : "+v"(tid_), "+v"(urow), "+v"(c), "+v"(srow), "+v"(gofs));
        const int tid = tid_, lane = tid & 63;
        const int left0 = nrows - urow;                  // rows q with 21 q < left0 exist
        const unsigned gofs_m = precond == 0 || lane == 63 ? gofs : 3u * gofs;
        const int lofs = 3 * (urow - row0) + c;          // in T entries of the rows' vectors
        // The previous iteration's |r|^2 and r.z (and the coarse correction's sums of r) are collected by
        // waves 0-3; meanwhile waves 4-7 wait for the few update workgroups whose z this one reads, and
        // read it.
        T zf[GF][3] = {};
        if (wave < 4) {
          if (!first) {
            double v[2];
            if (it == 0) {  // left by the launch before
              v[0] = v[1] = 0.0;
              for (int i = tid; i < NB; i += 256) {
                v[0] += gbl(rec()->part_rr)[i];
                v[1] += gbl(rec()->part_rz)[i];
              }
            } else if (solo) {
              v[0] = v[1] = 0.0;
              for (int i = tid; i < NU; i += 256) {
                v[0] += lp[nq + i];
                v[1] += lp[nq + nu + i];
              }
            } else {
              poll_sums<2>(rs_w, wprev, NX, tid, tag - 1u, &sh_failed, v);
            }
            const double s = wave_sum2(v[0], v[1]);
            if ((lane & 31) == 0) red[0][lane >> 5][wave] = s;
            if (coarse) {
              for (int k = 2; k < 5; k++) {
                double g[1] = {0.0};
                if (it == 0) {
                  for (int i = tid; i < NB; i += 256) g[0] += gbl(rec()->part_upd_g)[(size_t)(k - 2) * NB + i];
                } else if (solo) {
                  for (int i = tid; i < NU; i += 256) g[0] += lp[nq + k * nu + i];
                } else {
                  poll_sums<1>(rs_w, wprev + 16u * (unsigned)(k * NX), NX, tid, tag - 1u, &sh_failed, g);
                }
                const double gs = wave_sum(g[0]);
                if (lane == 0) red[0][k][wave] = gs;
              }
            }
          }
        } else if (nf > 0) {
          if (it > 0)
            for (int i = lane; i < nneed; i += 64) {
              const unsigned o[1] = {wprev + 16u * need[i]};
              double v[1];
              if (!poll_words<1>(rs_w, o, tag - 1u, v)) sh_failed = 1;
            }
          asm volatile("" ::: "memory");
          if (kF32) {
            for (int k = tid - 256; k < nf; k += 256 * GF) {
#pragma unroll
              for (int j = 0; j < GF; j++)
                ld_vertex(rs_z, 3u * ts * (unsigned)clist[foreign(min(k + 256 * j, nf - 1))], zf[j]);
#pragma unroll
              for (int j = 0; j < GF; j++) {
                const float4 q = make_float4((float)zf[j][0], (float)zf[j][1], (float)zf[j][2], 0.f);
                *(float4*)(lds + ZS * foreign(min(k + 256 * j, nf - 1))) = q;
              }
            }
          } else {
#pragma unroll
            for (int j = 0; j < GF; j++)
              if (256 * j < nf)
                ld_vertex(rs_z, 3u * ts * (unsigned)clist[foreign(min(tid - 256 + 256 * j, nf - 1))], zf[j]);
          }
        }
        __syncthreads();
        if (sh_failed) {
          done = 1;
          status = 2;
          break;
        }
        double beta = 0.0;
        if (!first) {
          double tot[5];
#pragma unroll
          for (int k = 0; k < 5; k++) {
            tot[k] = 0.0;
            if (k < 2 || coarse) {
#pragma unroll
              for (int w = 0; w < 4; w++) tot[k] += red[0][k][w];
              tot[k] = uniform_f(tot[k]);
            }
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
          if (not_finite(rrv) || !(rz == rz)) {
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
        if (!kF32) {  // p = z + beta p_old at every column (the own rows' z is in Tv)
          if (wave >= 4) {
#pragma unroll
            for (int j0 = 0; j0 < GF; j0 += 2) {
              if (256 * j0 >= nf) break;
              T pv[2][3];
              int k[2];
#pragma unroll
              for (int j = 0; j < 2; j++) {
                k[j] = tid - 256 + 256 * (j0 + j);
                const T* q = (const T*)(lds + ZS * foreign(min(k[j], nf - 1)));
#pragma unroll
                for (int e = 0; e < 3; e++) pv[j][e] = q[e];
              }
#pragma unroll
              for (int j = 0; j < 2; j++)
                if (k[j] < nf) {
                  T* q = (T*)(lds + ZS * foreign(k[j]));
#pragma unroll
                  for (int e = 0; e < 3; e++) q[e] = first ? zf[j0 + j][e] : fma(bt, pv[j][e], zf[j0 + j][e]);
                }
            }
            for (int k = tid - 256 + 256 * GF; k < nf; k += 256) {
              T v[3];
              ld_vertex(rs_z, 3u * ts * (unsigned)clist[foreign(k)], v);
              T* q = (T*)(lds + ZS * foreign(k));
#pragma unroll
              for (int e = 0; e < 3; e++) q[e] = first ? v[e] : fma(bt, q[e], v[e]);
            }
          } else {
            T* q = (T*)(lds + ZS * flo);
            const T* zs = Tv + 3 * (ua - row0);
            for (int i = tid; i < 3 * nown; i += 4 * 256) {
              T pv[4], zv[4];
#pragma unroll
              for (int j = 0; j < 4; j++) {
                const int k = min(i + 256 * j, 3 * nown - 1);
                pv[j] = q[k];
                zv[j] = zs[k];
              }
#pragma unroll
              for (int j = 0; j < 4; j++)
                if (j == 0 || i + 256 * j < 3 * nown) q[i + 256 * j] = first ? zv[j] : fma(bt, pv[j], zv[j]);
            }
          }
          __syncthreads();
        }
        // A times those entries, slice by slice, into Sv
        {
          T s0 = T(0), s1 = T(0), s2 = T(0), d0 = T(0), d1 = T(0), d2 = T(0);
          // the slice sums' place: the component and row this lane writes, in bytes
          const int scomp = H == 16 ? min(lane >> 4, 2) : H == 32 ? lane >> 5 : 0;
          unsigned so = (unsigned)off_s + ts * (unsigned)(3 * srow + scomp);
          int orow = srow;
          auto own_entry = [&]() {  // FP32: the row's own z, which its columns are relative to
            if (kF32) {
              const float4 q = *(const float4*)((char*)zown + ZS * min(orow, nrl - 1));
              d0 = (T)q.x;
              d1 = (T)q.y;
              d2 = (T)q.z;
            }
          };
          auto gather = [&](unsigned o, T(&v)[3]) {
            if (kF32) {
              const float4 q = *(const float4*)(lds + o);
              v[0] = (T)q.x;
              v[1] = (T)q.y;
              v[2] = (T)q.z;
            } else {
              const T* q = (const T*)(lds + o);
              v[0] = q[0];
              v[1] = q[1];
              v[2] = q[2];
            }
          };
          auto accumulate = [&](const T(&a)[9], const T(&v)[3]) {
            const T p0v = kF32 ? v[0] - d0 : v[0], p1v = kF32 ? v[1] - d1 : v[1], p2v = kF32 ? v[2] - d2 : v[2];
            s0 = row3(s0, a[0], a[1], a[2], p0v, p1v, p2v);
            s1 = row3(s1, a[3], a[4], a[5], p0v, p1v, p2v);
            s2 = row3(s2, a[6], a[7], a[8], p0v, p1v, p2v);
          };
          // the lanes of a row add their sums (i ^ 16 first, then i ^ 32), several components at once
          auto finish_slice = [&]() {
            if (H == 16) {
              const T a = swap_add<SWAP16>(s0, s1), b = swap_add<SWAP16>(s2, s2);
              *(T*)(lds + so) = swap_add<SWAP32>(a, b);
            } else if (H == 32) {
              *(T*)(lds + so) = swap_add<SWAP32>(s0, s1);
              const T b = swap_add<SWAP32>(s2, s2);
              if (scomp == 0) *(T*)(lds + so + 2 * ts) = b;
            } else {
              T* q = (T*)(lds + so);
              q[0] = s0;
              q[1] = s1;
              q[2] = s2;
            }
            s0 = s1 = s2 = T(0);
            so += 3 * ts * H * kResWaves;
            orow += H * kResWaves;
            own_entry();
          };
          own_entry();
          // the first streamed steps' values arrive during the others (BIG: past the last one, nothing is read)
          T sa9[ND][9] = {};
          unsigned slot = 0;
          int kj = str_cj;
          auto fetch = [&](T(&a)[9], int k) {
            size_t ns_ = ns;
            asm volatile("" : "+s"(ns_));
            if constexpr (BIG) {
              const unsigned o = k < nrest ? ts * slot : 0x7ffff000u;
#pragma unroll
              for (int e = 0; e < 9; e++) a[e] = buf_ld<T>(rs_a, o, (int)((unsigned)e * ts * (unsigned)ns_));
            } else {
#pragma unroll
              for (int e = 0; e < 9; e++) a[e] = ld_off(A + e * ns_, ts * slot);
            }
            slot += 64;
            if (k < nrest && ((ends >> (NR + k)) & 1) && ++kj < nslw)
              slot = (unsigned)(__builtin_amdgcn_readlane(l_beg, kj) + lane);
          };
          if (nlds < nrest) {
            slot = (unsigned)(__builtin_amdgcn_readlane(l_beg, str_cj) + 64 * str_cs + lane);
#pragma unroll
            for (int d = 0; d < ND; d++) fetch(sa9[d], nlds + d);
          }
          // the register steps in groups whose gathers are issued together (those past the wave's
          // last step multiply zeros)
          constexpr int G = kF32 ? 4 : 3;
#pragma unroll
          for (int k0 = 0; k0 < NR; k0 += G) {
            if (k0 < steps) {
              T v[G][3];
#pragma unroll
              for (int k = k0; k < k0 + G && k < NR; k++)
                gather((k & 1) ? ix[k >> 1] >> 16 : ix[k >> 1] & 0xffffu, v[k - k0]);
#pragma unroll
              for (int k = k0; k < k0 + G && k < NR; k++) {
                accumulate(m[k], v[k - k0]);
                if ((ends >> k) & 1) finish_slice();
              }
            }
          }
          for (int k = 0; k < nlds; k++) {
            T a[9], v[3];
#pragma unroll
            for (int e = 0; e < 9; e++) a[e] = ml[(9 * k + e) * 64 + lane];
            gather(idxr[64 * (rest_base + k) + lane], v);
            accumulate(a, v);
            if ((ends >> (NR + k)) & 1) finish_slice();
          }
          for (int k0 = nlds; k0 < nrest; k0 += ND) {
#pragma unroll
            for (int d = 0; d < ND; d++) {
              const int k = k0 + d;
              if (d == 0 || k < nrest) {
                T v[3];
                gather(idxr[64 * (rest_base + k) + lane], v);
                accumulate(sa9[d], v);
                if (BIG || k + ND < nrest) fetch(sa9[d], k + ND);
                if ((ends >> (NR + k)) & 1) finish_slice();
              }
            }
          }
        }
        // the first chunk's r, x and preconditioner, which the update needs: they arrive while p.t is awaited (past
        // the wave's chunks: rows that are not used, or past the end)
        T rv0[R], xv[R], m0[R], m1[R], m2[R];
        // this component's row of the chunk's aggregate inverse; with four row groups it costs more registers than the
        // latency is worth (24 served sessions 16.8 instead of 16.6 ms; 40^3 FP32 with two: 3.39 instead of 3.56)
        constexpr bool kInverse = kF32 && R == 2;
        T ai[3] = {};
        unsigned char pn[R];
        auto load = [&](unsigned go, unsigned gm, int left, int row, int ch) {
          if constexpr (kInverse)
            if (local && ch * 21 * R < nrows) {
              const unsigned o = ts * (unsigned)(9 * ch + 3 * c);
#pragma unroll
              for (int k = 0; k < 3; k++) ai[k] = ld_off(ainv, o + (unsigned)k * ts);
            }
#pragma unroll
          for (int q = 0; q < R; q++) {
            pn[q] = 1;
            if (local && 21 * q < left) pn[q] = ld_off(pinned, (unsigned)(row + 21 * q));
            rv0[q] = buf_ld<T>(rs_r, go + 63 * q * ts);
            xv[q] = buf_ld<T>(rs_x, go + 63 * q * ts);
            if (precond == 0) {
              m0[q] = buf_ld<T>(rs_m, gm + 63 * q * ts);
            } else {
              m0[q] = buf_ld<T>(rs_m, gm + 189 * q * ts);
              m1[q] = buf_ld<T>(rs_m, gm + 189 * q * ts + ts);
              m2[q] = buf_ld<T>(rs_m, gm + 189 * q * ts + 2 * ts);
            }
          }
        };
        // t and p of the rows, and p.t of each slice, L slices of the wave at a time
        for (int j0 = 0; j0 < nslw; j0 += L) {
          const int j = j0 + (lane >> sh);
          const int rl = srow + j * (H * kResWaves);
          double pt = 0.0;
          if (j < nslw && rl < nrl) {
            T s0 = Sv[3 * rl], s1 = Sv[3 * rl + 1], s2 = Sv[3 * rl + 2];
            if (kF32) {
              const float4 o = *(const float4*)((char*)zown + ZS * rl);
              T z0 = (T)o.x, z1 = (T)o.y, z2 = (T)o.z;
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
              const T* o = zown + 3 * rl;
              pt = dot3((double)o[0], (double)o[1], (double)o[2], (double)s0, (double)s1, (double)s2);
            }
          }
          // (the slices at the ends hold other workgroups' rows too)
          if (BIG && (row0 + rl < ua || row0 + rl >= ub)) pt = 0.0;
          pt = group_sum<H>(pt);
          if (j < nslw && (lane & (H - 1)) == 0) ptsl[wave + kResWaves * j] = pt;
        }
        __syncthreads();
        if (BIG) {
          if (wave == 0) {
            double s = 0.0;
            for (int i = lane; i < nsl; i += 64) s += ptsl[i];
            s = wave_sum(s);
            if (lane == 0) publish_word<SC>(rs_w, (tag & 1u) * npt + (unsigned)lb, s, tag);
          }
        } else if (split) {
          if (tid < nsl && (pubs[tid] >> 12) != 0) {
            const int e = pubs[tid], n = e >> 12;
            double v = n <= 4 ? ptsl[tid] : 0.0;
#pragma unroll
            for (int w = 1; w < 4; w++) v += w < n && n <= 4 ? ptsl[tid + w] : 0.0;
            publish_word<SC>(rs_w, (tag & 1u) * npt + (unsigned)(e & 0xfff), v, tag);
          }
        } else if (tid < max(nq, 1)) {
          double s = 0.0;
          if (nq > 0) {
#pragma unroll
            for (int w = 0; w < 4; w++) {
              const int sl = 4 * (q0 + tid) + w;
              s += sl < nslices ? ptsl[sl - sa] : 0.0;
            }
          }
          if (solo)
            lp[tid] = s;
          else
            publish_word<SC>(rs_w, (tag & 1u) * npt + (unsigned)(nq > 0 ? q0 + tid : qe), s, tag);
        }
        if (solo) __syncthreads();
        load(gofs, gofs_m, left0, urow, UC * u0 + wave);
        if (wave < 4) {
          double v[1] = {0.0};
          if (solo) {
            for (int i = tid; i < NQ; i += 256) v[0] += lp[i];
          } else if (split) {
            if (tid < np) {
              const unsigned m = apart[tid], o0 = 16u * (tag & 1u) * npt + 64u * (unsigned)tid;
              if (kF32) {
                const unsigned o[4] = {o0, o0 + (m & 2u) * 8u, o0 + (m & 4u) * 8u, o0 + (m & 8u) * 6u};
                double g[4];
                if (!poll_words<4>(rs_w, o, tag, g)) sh_failed = 1;
                v[0] = g[0];
#pragma unroll
                for (int j = 1; j < 4; j++)
                  if (m >> j & 1u) v[0] += g[j];
              } else {
                unsigned o[1] = {o0};
                double g[1];
                unsigned left = m | 1u;
                while (left) {  // (the others are usually there by the time the first one is)
                  const unsigned j = (unsigned)__ffs((int)left) - 1u;
                  o[0] = o0 + 16u * j;
                  if (!poll_words<1>(rs_w, o, tag, g)) sh_failed = 1;
                  v[0] += g[0];
                  left &= left - 1u;
                }
              }
            }
          } else {
            poll_sums<1>(rs_w, 16u * (tag & 1u) * npt, np, tid, tag, &sh_failed, v);
          }
          v[0] = wave_sum(v[0]);
          if (lane == 0) red[1][0][wave] = v[0];
        }
        __syncthreads();
        if (sh_failed) {
          done = 1;
          status = 2;
          break;
        }
        // alpha, then x, r and z of the own rows, chunk by chunk
        double ptt = 0.0;
#pragma unroll
        for (int w = 0; w < 4; w++) ptt += red[1][0][w];
        const T alpha = (T)(absNew / uniform_f(ptt));
        for (int cl = wave; cl < nch; cl += kResWaves) {
          const int ch = (cl - wave) * 21 * R;  // rows past the first chunk's
          const unsigned go = gofs + 3u * ts * (unsigned)ch;
          const int left = left0 - ch, lo = lofs + 3 * ch;
          T rq[R], zq[R];
          double rr2 = 0.0, rz = 0.0, gc = 0.0;
#pragma unroll
          for (int q = 0; q < R; q++) {
            T rv = T(0);
            if (21 * q < left) rv = fma(-alpha, Tv[lo + 63 * q], rv0[q]);
            const T r0 = __shfl(rv, lane - c, 64);
            const T r1 = __shfl(rv, lane - c + 1, 64);
            const T r2 = __shfl(rv, lane - c + 2, 64);
            rq[q] = rv;
            zq[q] = precond == 0 ? m0[q] * rv : fma(m2[q], r2, fma(m0[q], r0, m1[q] * r1));
          }
          if constexpr (kF32) {
            if (local) {
              if constexpr (kInverse)
                agg_apply<T, R>(ai, c, rq, pn, zq);
              else
                agg_correct<T, R>(ainv, UC * u0 + cl < (nrows + 21 * R - 1) / (21 * R) ? UC * u0 + cl : 0, c, rq, pn, zq);
            }
          }
#pragma unroll
          for (int q = 0; q < R; q++) {
            buf_st<SC>(rs_z, go + 63 * q * ts, zq[q]);
            if (21 * q < left) {
              rr2 = fma((double)rq[q], (double)rq[q], rr2);
              rz = fma((double)rq[q], (double)zq[q], rz);
              gc += (double)rq[q];
            }
          }
          const double v2 = wave_sum2(rr2, rz);
          if ((lane & 31) == 0) uw[(lane >> 5) * nch + cl] = v2;
          if (coarse) {
            const double g2 = wave_sum2(c == 0 ? gc : 0.0, c == 1 ? gc : 0.0), g = wave_sum(c == 2 ? gc : 0.0);
            if ((lane & 31) == 0) uw[(2 + (lane >> 5)) * nch + cl] = g2;
            if (lane == 0) uw[4 * nch + cl] = g;
          }
#pragma unroll
          for (int q = 0; q < R; q++) {
            buf_st<0>(rs_r, go + 63 * q * ts, rq[q]);
            if (21 * q < left) {
              const int l = lo + 63 * q;
              const T pv = kF32 ? Pv[l] : zown[l];
              buf_st<0>(rs_x, go + 63 * q * ts, fma(alpha, pv, xv[q]));
              if (kF32)
                zown[4 * (urow + ch + 21 * q - row0) + c] = zq[q];
              else
                Tv[l] = zq[q];
            }
          }
          if (cl + kResWaves < nch) {
            constexpr int step = kResWaves * 21 * R;
            load(go + 3u * ts * step, gofs_m + (precond == 0 ? 3u : 9u) * ts * (unsigned)(ch + step), left - step,
                 urow + ch + step, UC * u0 + cl + kResWaves);
          }
        }
        // z is complete before the sums that announce it are published
        if (!solo) __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (BIG) {
          if (wave < nval) {
            double s = 0.0;
            for (int i = lane; i < nch; i += 64) s += uw[wave * nch + i];
            s = wave_sum(s);
            if (lane == 0) publish_word<SC>(rs_w, 2u * npt + (5u * (tag & 1u) + (unsigned)wave) * (unsigned)NX + (unsigned)lb, s, tag);
            if (it == iters - 1) {  // the next launch adds all NB of them
              const auto J = rec();
              auto dst = gbl(wave == 0 ? J->part_rr : wave == 1 ? J->part_rz : J->part_upd_g + (size_t)(wave - 2) * NB);
              for (int i = lb + W * lane; i < NB; i += 64 * W) dst[i] = lane == 0 ? s : 0.0;
            }
          }
        } else if (tid < nval * nu) {
          int kind = 0, ku = tid;  // the update sum this thread publishes
          for (; ku >= nu; kind++) ku -= nu;
          double s = 0.0;
#pragma unroll
          for (int w = 0; w < 4; w++) s += uw[kind * nch + 4 * ku + w];
          if (solo)
            lp[nq + kind * nu + ku] = s;
          else
            publish_word<SC>(rs_w, 2u * npt + (5u * (tag & 1u) + (unsigned)kind) * (unsigned)NU + (unsigned)(u0 + ku),
                         s, tag);
          if (it == iters - 1) {  // the next launch finishes this iteration from these
            const auto J = rec();
            auto dst = kind == 0 ? J->part_rr : kind == 1 ? J->part_rz : J->part_upd_g + (size_t)(kind - 2) * NU;
            gbl(dst)[u0 + ku] = s;
          }
        }
        if (solo) __syncthreads();
        first = false;
      }
      __syncthreads();
      if (!done)  // the solve goes on in another launch: its p and t
        for (int i = tid; i < 3 * nown; i += kResThreads) {
          const size_t g = 3 * (size_t)ua + i;
          const int l = 3 * (ua - row0) + i;
          gbl((T*)rec()->p0)[g] = kF32 ? Pv[l] : zown[l];
          if (kF32) gbl((T*)rec()->t)[g] = Tv[l];
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
        ctl->res_work += (unsigned)it;
        ctl->res_runs += 1u;
        ctl->res_epoch = epoch + 2u + (unsigned)it;
      }
    }
  }
  // the last workgroup to leave clears the instance's meeting point (ONE: if all W of them came; see the kernel)
  __syncthreads();
  if (tid == 0) {
    if (sh_failed) {
      __hip_atomic_fetch_or(arr, kLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_s_waitcnt(0);  // before it counts as having left
    }
    auto ex = (HOBAK_GLOBAL int*)&ctl->res_exit;
    if (__hip_atomic_fetch_add(ex, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == W - 1) {
      const int v = __hip_atomic_load(arr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (v & kAbort) ctl->res_abort += 1;
      if ((v & kAbort) == kLate) ctl->res_late += 1;
      if (v & kLost) ctl->res_lost = 1;
      __hip_atomic_store(arr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(ex, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// b: boff[i] counts the workgroups of instance i.  tickets: [0] the next ticket, [1] workgroups done;
// both zero between launches.
template <typename T, int R, int H, bool BIG>
__global__ __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void cg_resident_kernel(
    Batch b, int* tickets, int iters) {
  extern __shared__ __align__(16) char lds[];
  __shared__ int sh_ticket;
  if (threadIdx.x == 0)
    sh_ticket = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  int lb, W;
  const HOBAK_GLOBAL InstDev* I =
      uptr((const InstDev*)seg_find(b, __builtin_amdgcn_readfirstlane(sh_ticket), lb, W));
  resident_solve<T, R, H, BIG, false>(I, uniform_i(lb), uniform_i(W), iters, lds);
  if (threadIdx.x == 0 &&
      __hip_atomic_fetch_add(tickets + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == b.total - 1) {
    __hip_atomic_store(tickets, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(tickets + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The arguments of cg_resident_die_kernel, read anew from the argument segment: what its end needs is not held in
// scalar registers through the solve.
struct DieArgs {
  Batch b;
  int* tickets;
};
__device__ __forceinline__ const __attribute__((address_space(4))) DieArgs* late_args() {
  auto a = (const __attribute__((address_space(4))) DieArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}

// The same for up to eight instances, instance i on die `first` + i (mod 8) alone: the grid holds as many workgroups for each die as
// the largest instance takes, and those past an instance's, or of a die without one, leave at once.
// tickets: [0] workgroups done, [1 + i] instance i's next ticket; all zero between launches.
template <typename T, int R, int H>
__global__ __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void cg_resident_die_kernel(
    Batch b, int* tickets, int iters, int first) {
  extern __shared__ __align__(16) char lds[];
  __shared__ int sh_ticket;
  const int i = __builtin_amdgcn_readfirstlane((die_of_wave() - first) & (kResDies - 1));
  if (i < b.n) {
    const int W = uniform_i(b.n == 1 ? b.total : gbl(b.boff)[i + 1] - gbl(b.boff)[i]);
    if (threadIdx.x == 0)
      sh_ticket = __hip_atomic_fetch_add(tickets + 1 + i, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int lb = uniform_i(sh_ticket);
    if (lb < W) {
      const HOBAK_GLOBAL InstDev* I = uptr(b.n == 1 ? b.one : gbl(b.inst)[i]);
      resident_solve<T, R, H, false, true>(I, lb, W, iters, lds);
    }
  }
  if (threadIdx.x != 0) return;
  __builtin_amdgcn_s_waitcnt(0);  // what this workgroup did to its meeting point is done
  const auto args = late_args();
  const auto t = gbl(args->tickets);
  if (__hip_atomic_fetch_add(t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (int)gridDim.x - 1) return;
  // the grid's last workgroup: an instance whose die got too few workgroups is untouched, and its meeting point
  // holds what those that came left there
  const int n = args->b.n;
  for (int k = 0; k < n; k++) {
    const int W = n == 1 ? args->b.total : gbl(args->b.boff)[k + 1] - gbl(args->b.boff)[k];
    if (__hip_atomic_load(t + 1 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= W) continue;
    auto ctl = ctl_of(gbl(n == 1 ? args->b.one : gbl(args->b.inst)[k]));
    if (ctl->sc[0].done) continue;
    ctl->res_abort += 1;
    ctl->res_late += 1;
    __hip_atomic_store((HOBAK_GLOBAL int*)&ctl->res_arrive, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store((HOBAK_GLOBAL int*)&ctl->res_exit, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int k = 0; k <= kResDies; k++) __hip_atomic_store(t + k, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T, int R, int H, bool BIG>
hipError_t resident_rh(const Batch& b, int* tickets, int iters, hipStream_t s) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&cg_resident_kernel<T, R, H, BIG>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kResLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((cg_resident_kernel<T, R, H, BIG>), dim3(b.total), dim3(kResThreads), kResLds, s, b, tickets,
                     iters);
  return hipGetLastError();
}
template <typename T, int R, int H>
hipError_t resident_die(const Batch& b, int first, int wgs, int* tickets, int iters, hipStream_t s) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&cg_resident_die_kernel<T, R, H>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kResLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((cg_resident_die_kernel<T, R, H>), dim3(kResDies * wgs), dim3(kResThreads), kResLds, s, b, tickets,
                     iters, first);
  return hipGetLastError();
}
template <typename T, int R>
hipError_t resident_die_r(const Batch& b, int shift, int first, int wgs, int* tickets, int iters, hipStream_t s) {
  switch (shift) {
    case 4: return resident_die<T, R, 16>(b, first, wgs, tickets, iters, s);
    case 5: return resident_die<T, R, 32>(b, first, wgs, tickets, iters, s);
    case 6: return resident_die<T, R, 64>(b, first, wgs, tickets, iters, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename T, int R, bool BIG>
hipError_t resident_r(const Batch& b, int shift, int* tickets, int iters, hipStream_t s) {
  switch (shift) {
    case 4: return resident_rh<T, R, 16, BIG>(b, tickets, iters, s);
    case 5: return resident_rh<T, R, 32, BIG>(b, tickets, iters, s);
    case 6: return resident_rh<T, R, 64, BIG>(b, tickets, iters, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

size_t resident_words(int nb_spmv, int nb_upd) {
  const size_t npt = nb_spmv <= kSplitMax ? 4 * (size_t)(nb_spmv + 1) : 0;
  return 4 * std::max(npt, (size_t)nb_spmv + nb_upd) + 20 * (size_t)nb_upd;
}
bool resident_layout(int shift, int groups, int nb_upd) {
  return shift >= 4 && shift <= 6 && (groups == 2 || groups == 4) && nb_upd <= kResMaxUpd;
}
bool resident_layout_big(int shift, int groups, int nb_upd, int wgs) {
  return shift >= 4 && shift <= 6 && (groups == 2 || groups == 4) && wgs <= std::min(nb_upd, 256);
}

template <typename T>
hipError_t launch_cg_resident(const Batch& b, int shift, int groups, bool big, int* tickets, int iters, hipStream_t s) {
  if (b.total <= 0) return hipSuccess;
  if constexpr (sizeof(T) < sizeof(double)) {
    if (big) return groups == 2 ? resident_r<T, 2, true>(b, shift, tickets, iters, s) : resident_r<T, 4, true>(b, shift, tickets, iters, s);
  }
  if (big) return hipErrorInvalidValue;
  switch (groups) {
    case 2: return resident_r<T, 2, false>(b, shift, tickets, iters, s);
    case 4: return resident_r<T, 4, false>(b, shift, tickets, iters, s);
    default: return hipErrorInvalidValue;
  }
}
template <typename T>
hipError_t launch_cg_resident_die(const Batch& b, int shift, int groups, int first, int wgs, int* tickets, int iters,
                                  hipStream_t s) {
  if (b.n < 1 || b.n > kResDies || wgs < 1) return hipErrorInvalidValue;
  switch (groups) {
    case 2: return resident_die_r<T, 2>(b, shift, first, wgs, tickets, iters, s);
    case 4: return resident_die_r<T, 4>(b, shift, first, wgs, tickets, iters, s);
    default: return hipErrorInvalidValue;
  }
}
template hipError_t launch_cg_resident_die<double>(const Batch&, int, int, int, int, int*, int, hipStream_t);
template hipError_t launch_cg_resident_die<float>(const Batch&, int, int, int, int, int*, int, hipStream_t);
template hipError_t launch_cg_resident<double>(const Batch&, int, int, bool, int*, int, hipStream_t);
template hipError_t launch_cg_resident<float>(const Batch&, int, int, bool, int*, int, hipStream_t);

}  // namespace hobak
