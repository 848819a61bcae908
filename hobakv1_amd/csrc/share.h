// How the contexts of one process share a device's compute units in the resident PCG.
//
// The workgroups of a resident launch wait for each other, so two launches that each hold part of the compute units they
// need would both wait until they give up (0.2 s each time; four contexts of 303,242, 68,921, 9,261 and 1,331
// vertices stepping in four threads took up to 1.4 s for a step).  A context therefore claims the compute units of
// its launches, by die, while they are queued or running.  Where they do not fit beside those of others its
// stream first waits for those: claims are made one at a time, so a launch only ever waits for earlier ones.
//
// A launch holds its compute units for a whole solve, which a context with a small instance would wait for each
// time.  Of contexts that were in each other's way lately, one whose launches take longer than another's therefore
// takes turns of about the other's length.  (Contexts that one thread uses in turn never are.)
//
// Groups of the two-kernel form wait for nobody, but their launches get only the compute units that resident ones leave,
// between launches or beside them (57x64x50 in FP64 beside a 40^3 stepper: 200 ms a step, 60 before the resident PCG).
// A context that queues groups therefore publishes an event behind each, and a launch that takes more than a
// quarter of the device beside such a context first lets it run two groups, and takes a short turn.  So does, without the
// wait, a launch that leaves no compute unit while another context is in a call of short kernels.
#pragma once
#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

namespace hobak {

constexpr int kShareDies = 8;

// One context's part of a device.
struct Claim {
  void* done = nullptr;      // the event behind its last launch
  int use[kShareDies] = {};  // compute units on each die
  double ms = 0.0;           // what its launches take, roughly
  double met_s = -1e9;       // when it last did not fit beside another, or another beside it
  bool live = false;         // its launches are queued or running
  std::vector<void*> groups; // the events behind its groups of the two-kernel form in this tick ...
  size_t passed = 0;         // ... of which this many are known to have run
  double groups_s = -1e9;    // when another's launch last found any
  std::atomic<int> calls{0}; // calls in progress that only launch short kernels (forces, stiffness)
  double calls_s = -1e9;     // when a launch that filled the device last found any
};

constexpr double kShareLatelyS = 0.05;  // contexts that were in each other's way within this time are expected to be again
constexpr double kShareTurnMs = 2.0;    // the shortest turn: a launch's set-up and the host's part take 0.1 ms ...
constexpr double kGroupsTurnMs = 1.0;   // ... and beside groups, of which two take 0.4 ms (40^3) to 2 ms (57x64x50)
constexpr size_t kGroupsAhead = 2;

struct Share {
  std::mutex mu;               // held while a claim is made and its launches are queued
  std::vector<Claim*> claims;  // of every context on the device

  // The compute units that live claims of others hold on each die; false if there are none.
  bool held(const Claim* mine, int (&sum)[kShareDies]) const {
    bool any = false;
    for (int& u : sum) u = 0;
    for (const Claim* c : claims)
      if (c != mine && c->live) {
        any = true;
        for (int d = 0; d < kShareDies; d++) sum[d] += c->use[d];
      }
    return any;
  }
  // Whether `use` fits beside `sum` (on `per_die` compute units a die).
  static bool fits(const int (&sum)[kShareDies], const int (&use)[kShareDies], int per_die) {
    for (int d = 0; d < kShareDies; d++)
      if (sum[d] + use[d] > per_die) return false;
    return true;
  }
  // `mine` does not fit beside the live claims of others.
  void meets(Claim* mine, double now_s) {
    for (Claim* c : claims)
      if (c == mine || c->live) c->met_s = now_s;
  }
  // The longest a turn of `mine` should take: no limit (0), or as long as the shortest of the others it met.
  double turn_ms(const Claim* mine, double now_s) const {
    double ms = 0.0;
    if (now_s - mine->met_s < kShareLatelyS)
      for (const Claim* c : claims)
        if (c != mine && now_s - c->met_s < kShareLatelyS) ms = ms > 0.0 ? std::min(ms, c->ms) : c->ms;
    return ms > 0.0 ? std::max(ms, kShareTurnMs) : 0.0;
  }
  // Whether `use` is so much of the device (of `per_die` compute units a die) that others' groups need turns.
  static bool large(const int (&use)[kShareDies], int per_die) {
    int sum = 0;
    for (int u : use) sum += u;
    return 4 * sum > kShareDies * per_die;
  }
  static bool fills(const int (&use)[kShareDies], int per_die) {
    return *std::min_element(use, use + kShareDies) >= per_die;
  }
  // Whether another context is in a call of short kernels, or was lately.
  bool calls_lately(const Claim* mine, double now_s) {
    bool any = false;
    for (Claim* c : claims) {
      if (c == mine) continue;
      if (c->calls.load(std::memory_order_relaxed) > 0) c->calls_s = now_s;
      any |= now_s - c->calls_s < kShareLatelyS;
    }
    return any;
  }
  // Whether another context has groups queued, or had when a launch lately looked.
  bool groups_lately(const Claim* mine, double now_s) {
    bool any = false;
    for (Claim* c : claims) {
      if (c == mine) continue;
      if (!c->groups.empty()) c->groups_s = now_s;
      any |= now_s - c->groups_s < kShareLatelyS;
    }
    return any;
  }
  // The die on which to put the first of `n` instances that take wgs[i] compute units of successive dies: where
  // the fullest die is emptiest; -1 if they fit on none.
  static int first_die(const int (&sum)[kShareDies], const int* wgs, int n, int per_die) {
    int best = -1, least = per_die + 1;
    for (int first = 0; first < kShareDies; first++) {
      int full = 0, use[kShareDies];
      std::copy(sum, sum + kShareDies, use);
      for (int i = 0; i < n; i++) use[(first + i) % kShareDies] += wgs[i];
      for (int u : use) full = std::max(full, u);
      if (full < least) {
        least = full;
        best = first;
      }
    }
    return best;
  }
};

}  // namespace hobak
