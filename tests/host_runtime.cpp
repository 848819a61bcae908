// A HIP runtime for tests of the step engine's host code (api.hip) on the CPU: device memory is host memory, and a
// launch runs a stand-in for the kernel that keeps the PCG's bookkeeping only.  A solve takes the sweeps and
// iterations per sweep that the test gives for the instance's vertex count, and a resident launch does with an
// instance what the test says (Outcome).  Every launch of interest is written to a log the test reads.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../hobakv1_amd/csrc/kernels.h"

using namespace hobak;

namespace {
enum Outcome { RUNS = 0, MISFIT = 1, LATE = 2, LOST = 3 };
struct Script {
  int sweeps = 1, iters = 10;
  int outcome[3] = {RUNS, RUNS, RUNS};  // over the device, on one die, on every compute unit
};
std::map<int, Script> g_script;  // by vertex count
std::map<const void*, std::string>& kernel_names() {  // filled by other files' static initialisers
  static std::map<const void*, std::string> names;
  return names;
}
std::string g_log;
int g_device = 0, g_wrong_device = 0, g_events = 0;

struct Stream {
  int device;
  bool capturing = false;
  std::vector<std::function<void()>> recorded;
};
typedef std::vector<std::function<void()>> Graph;

void log_line(const std::string& s) { g_log += s + "\n"; }
Stream* on(hipStream_t s) {
  Stream* st = (Stream*)s;
  if (st && st->device != g_device) g_wrong_device++;
  return st;
}
const InstDev* inst(const Batch& b, int i) { return b.n == 1 ? b.one : b.inst[i]; }
bool has(const std::string& name, const char* kernel) { return name.find(kernel) != std::string::npos; }

// one PCG iteration of every instance whose solve is running
void iterate(const Batch& b) {
  for (int i = 0; i < b.n; i++) {
    Ctl* c = ctl_of(inst(b, i));
    if (c->sc[0].done) continue;
    c->sc[0].first = 0;
    if (++c->sc[0].iters >= g_script[inst(b, i)->nv].iters) c->sc[0].done = 1;
  }
}

void resident(const Batch& b, int form, int iters) {
  for (int i = 0; i < b.n; i++) {
    const InstDev* I = inst(b, i);
    Ctl* c = ctl_of(I);
    if (c->sc[0].done) continue;
    const Script& s = g_script[I->nv];
    const int what = s.outcome[form];
    if (what == LOST) {
      c->res_lost = 1;
      c->res_runs += 1;
      continue;
    }
    if (what != RUNS) {
      c->res_abort += 1;
      if (what == LATE) c->res_late += 1;
      continue;
    }
    const int k = std::min(iters, s.iters - c->sc[0].iters);
    c->sc[0].iters += k;
    c->sc[0].first = 0;
    if (c->sc[0].iters >= s.iters) c->sc[0].done = 1;
    c->res_work += (unsigned)k;
    c->res_runs += 1;
  }
}

template <typename T>
T arg(void** a, int i) {
  T v;
  std::memcpy(&v, a[i], sizeof(T));
  return v;
}

// What a launch does when the stream reaches it.
std::function<void()> stand_in(const std::string& name, void** a) {
  if (has(name, "cg_init_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    const int gate = arg<int>(a, 2);
    return [=] {
      for (int i = 0; i < b.n; i++) {
        Ctl* c = ctl_of(inst(b, i));
        if (gate && !(c->phase == PHASE_SOLVING && c->sc[0].done)) continue;
        if (!gate) c->rs = RefineState{};
        c->sc[0] = CgScalars{};
        c->sc[0].first = 1;
        if (!gate) c->res_lost = 0;
        c->phase = PHASE_SOLVING;
      }
    };
  }
  if (has(name, "cg_spmv_kernel") || has(name, "cg_spmv_p_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    return [=] {
      log_line("spmv " + std::to_string(b.n));
      for (int i = 0; i < b.n; i++)
        if (!ctl_of(inst(b, i))->sc[0].done) ctl_of(inst(b, i))->spmv_work += 1;
    };
  }
  if (has(name, "cg_update_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    return [=] { iterate(b); };
  }
  if (has(name, "cg_resident_kernel") || has(name, "cg_resident_die_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    const int iters = arg<int>(a, 2);
    const int form = has(name, "die") ? 1 : has(name, "Lb1E") ? 2 : 0;  // template argument BIG == true
    return [=] {
      log_line(std::string(form == 0 ? "device " : form == 1 ? "die " : "big ") + std::to_string(b.n) + " iters " +
               std::to_string(iters));
      resident(b, form, iters);
    };
  }
  if (has(name, "finish_check_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    const int refine = arg<int>(a, 1);
    return [=] {
      for (int i = 0; i < b.n; i++) {
        Ctl* c = ctl_of(inst(b, i));
        if (c->phase == PHASE_SOLVING && c->res_lost) {
          c->sc[0].done = 1;
          c->phase = PHASE_FINISHED;
          continue;
        }
        if (!(c->phase == PHASE_SOLVING && c->sc[0].done)) continue;
        if (refine) {
          c->rs.inner_iters += c->sc[0].iters;
          if (++c->rs.sweeps == 1) c->rs.first_iters = c->sc[0].iters;
          c->rs.done = c->rs.sweeps >= g_script[inst(b, i)->nv].sweeps;
        }
        if (!refine || c->rs.done) c->phase = PHASE_FINISHED;
      }
    };
  }
  if (has(name, "status_kernel")) {
    const Batch b = arg<Batch>(a, 0);
    InstStatus* out = arg<InstStatus*>(a, 1);
    return [=] {
      log_line("status " + std::to_string(b.n));
      for (int i = 0; i < b.n; i++) {
        const Ctl* c = ctl_of(inst(b, i));
        InstStatus o = {};
        o.phase = c->phase;
        o.iters = c->sc[0].iters;
        o.inner_total = c->rs.inner_iters;
        o.sweeps = c->rs.sweeps;
        o.ref_done = c->rs.done;
        o.first_iters = inst(b, i)->refine ? c->rs.first_iters : c->sc[0].iters;
        o.spmv_work = c->spmv_work;
        o.res_work = c->res_work;
        o.res_abort = c->res_abort;
        o.res_late = c->res_late;
        o.res_lost = c->res_lost;
        o.res_runs = c->res_runs;
        out[i] = o;
      }
    };
  }
  if (has(name, "state_kernel")) return [=] { log_line("state"); };
  if (has(name, "begin_step_kernel")) return [=] { log_line("begin"); };
  return [] {};
}

hipError_t launch(const void* f, void** a, hipStream_t s) {
  Stream* st = on(s);
  auto run = stand_in(kernel_names()[f], a);
  if (st && st->capturing)
    st->recorded.push_back(run);
  else
    run();
  return hipSuccess;
}
}  // namespace

extern "C" {
// -- the test's side
void fake_script(int nv, int sweeps, int iters, int device, int die, int big) {
  g_script[nv] = Script{sweeps, iters, {device, die, big}};
}
const char* fake_log() { return g_log.c_str(); }
void fake_clear() {
  g_log.clear();
  g_wrong_device = 0;
}
void fake_reset() {
  fake_clear();
  g_script.clear();
  g_device = 0;
}
int fake_wrong_device() { return g_wrong_device; }

// -- the runtime's side
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernel_names()[f] = name;
}
static thread_local struct {
  dim3 g, b;
  size_t sh;
  hipStream_t s;
} t_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  t_call.g = g, t_call.b = b, t_call.sh = sh, t_call.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
  *g = t_call.g, *b = t_call.b, *sh = t_call.sh, *s = t_call.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** a, size_t, hipStream_t s) { return launch(f, a, s); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** a, size_t, hipStream_t s, hipEvent_t e, hipEvent_t, int) {
  if (e) log_line("sample");
  return launch(f, a, s);
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  g_device = d;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char room[1 << 16];
  *p = room;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  (void)q;
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)(intptr_t)++g_events;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  log_line("after");
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t) new Stream{g_device};
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete (Stream*)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  log_line("wait");
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  ((Stream*)s)->capturing = true;
  ((Stream*)s)->recorded.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  ((Stream*)s)->capturing = false;
  *g = (hipGraph_t) new Graph(((Stream*)s)->recorded);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t) new Graph(*(Graph*)g);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (Graph*)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete (Graph*)e;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  on(s);
  for (auto& f : *(Graph*)e) f();
  return hipSuccess;
}
int roctxRangePushA(const char*) { return 0; }
int roctxRangePop() { return 0; }
}
