// A HIP runtime for CPU tests of the host code: device memory is host memory,
// kernels do nothing, and every launch is checked.  A pointer argument has to
// point into a live allocation; one may be null only if it was null in some
// launch of that kernel while `learn` was on.  Captured launches are checked
// again at every replay.  Memory starts as doubles of value 1 and is never
// reused, so stale pointers show.  The k-th next hipMalloc can be made to fail.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "../../tmr_amd/csrc/forest.h"
#include "../../tmr_amd/csrc/kernels.h"

namespace {
struct Block {
  size_t n;
  bool live;
  int kind;  // hipMemoryType
};
struct Kernel {
  std::string name;
  std::vector<std::string> args;
};
struct Launch {
  const Kernel *k;
  std::vector<const void *> ptr;   // pointer arguments (null where not one)
  std::vector<const void *> plan;  // those inside a SegPlan
};
std::map<uintptr_t, Block> mem;
std::map<const void *, Kernel> kernels;
std::map<std::string, std::set<uint64_t>> nulls;
std::vector<std::string> bad;
std::vector<Launch> *capture = nullptr;
int fail_in = 0, allocs = 0;
bool learn = true;
size_t max_lds = 160 * 1024;
struct {
  dim3 grid, block;
  size_t sh;
  hipStream_t st;
} call;

// 0 null, 1 live, 2 anything else
int state(const void *p) {
  if (!p) return 0;
  auto it = mem.upper_bound((uintptr_t)p);
  if (it == mem.begin()) return 2;
  --it;
  return it->second.live && (uintptr_t)p <= it->first + it->second.n ? 1 : 2;
}

void run(const Launch &l) {
  uint64_t mask = 0;
  for (size_t i = 0; i < l.ptr.size(); i++) {
    if (l.k->args[i].back() != '*') continue;
    const int s = state(l.ptr[i]);
    if (s == 0) mask |= uint64_t(1) << i;
    if (s == 2) bad.push_back(l.k->name + ": argument " + std::to_string(i) + " is not live");
  }
  for (const void *p : l.plan)
    if (state(p) != 1) bad.push_back(l.k->name + ": plan is not live");
  if (learn)
    nulls[l.k->name].insert(mask);
  else if (mask && !nulls[l.k->name].count(mask))
    bad.push_back(l.k->name + ": unexpected null arguments");
  // one iteration runs, then the solve has converged
  auto word = [&](size_t i, int v) {
    if (i < l.ptr.size() && l.ptr[i]) *(int *)l.ptr[i] = v;
  };
  if (l.k->name.find("k_b_tick") != std::string::npos) word(4, 1);
  if (l.k->name.find("k_b_finalize") != std::string::npos) word(11, 0);
}

hipError_t give(void **p, size_t n, int kind) {
  allocs++;
  if (fail_in > 0 && --fail_in == 0) return hipErrorOutOfMemory;
  const size_t m = (n + 64) / 8;
  double *d = (double *)malloc(8 * m);
  for (size_t i = 0; i < m; i++) d[i] = 1.0;
  mem[(uintptr_t)d] = {n, true, kind};
  *p = d;
  return hipSuccess;
}
hipError_t take(void *p) {
  if (!p) return hipSuccess;
  auto it = mem.find((uintptr_t)p);
  if (it == mem.end() || !it->second.live) {
    bad.push_back("free of a pointer that is not live");
    return hipErrorInvalidValue;
  }
  it->second.live = false;
  return hipSuccess;
}
bool dead(const void *p) {
  auto it = mem.upper_bound((uintptr_t)p);
  if (it == mem.begin()) return false;
  --it;
  return !it->second.live && (uintptr_t)p < it->first + it->second.n;
}
}  // namespace

extern "C" {
void fake_fail_in(int k) { fail_in = k; }
int fake_allocs() { return allocs; }
void fake_learn(int on) { learn = on != 0; }
void fake_max_lds(int bytes) { max_lds = (size_t)bytes; }
int fake_bad(char *out, int n) {
  std::string s;
  for (size_t i = 0; i < bad.size() && i < 4; i++) s += bad[i] + "\n";
  strncpy(out, s.c_str(), n - 1);
  const int k = (int)bad.size();
  bad.clear();
  return k;
}

// linked with --wrap: the interpolation passes run on the host
int __wrap__ZN4tmrx6Forest27create_interpolation_deviceEPS0_RNS_9InterpCSREiPd(
    tmrx::Forest *f, tmrx::Forest *coarse, tmrx::InterpCSR &P, int, double *) {
  return f->create_interpolation(coarse, P);
}

hipError_t hipMalloc(void **p, size_t n) { return give(p, n, hipMemoryTypeDevice); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return give(p, n, hipMemoryTypeHost); }
hipError_t hipFree(void *p) { return take(p); }
hipError_t hipHostFree(void *p) { return take(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  if (n && (!d || !s || dead(d) || dead(s))) {
    bad.push_back("copy from or to memory that is not live");
    return hipErrorInvalidValue;
  }
  if (n) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void *d, int v, size_t n) {
  if (n && state(d) != 1) {
    bad.push_back("memset of memory that is not live");
    return hipErrorInvalidValue;
  }
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  memset(a, 0, sizeof(*a));
  auto it = mem.upper_bound((uintptr_t)p);
  if (state(p) != 1) return hipErrorInvalidValue;
  a->type = (hipMemoryType)(--it)->second.kind;
  return hipSuccess;
}

hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  return *v = (int)max_lds, hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof(*p));
  p->sharedMemPerBlock = max_lds;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) {
  return e == hipSuccess ? "success" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  return *s = (hipStream_t)malloc(1), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)malloc(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return capture = new std::vector<Launch>, hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)capture;
  capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *e = (hipGraphExec_t) new std::vector<Launch>(*(std::vector<Launch> *)g);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete (std::vector<Launch> *)g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t g) {
  return delete (std::vector<Launch> *)g, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t) {
  for (const Launch &l : *(std::vector<Launch> *)g) run(l);
  return hipSuccess;
}

void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  int st = 0;
  char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  Kernel k;
  const std::string s = st == 0 ? d : name;
  free(d);
  // the parameter list is the last parenthesised group
  const size_t close = s.rfind(')');
  size_t open = close;
  for (int depth = 0; open != std::string::npos; open--) {
    if (s[open] == ')') depth++;
    if (s[open] == '(' && --depth == 0) break;
  }
  k.name = s.substr(0, open);
  std::string a;
  int depth = 0;
  for (size_t i = open + 1; i <= close && open != std::string::npos; i++) {
    if ((s[i] == ',' && depth == 0) || i == close) {
      while (!a.empty() && a[0] == ' ') a.erase(0, 1);
      k.args.push_back(a);
      a.clear();
      continue;
    }
    if (s[i] == '<' || s[i] == '(') depth++;
    if (s[i] == '>' || s[i] == ')') depth--;
    a += s[i];
  }
  kernels[host] = k;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  call = {g, b, sh, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
  *g = call.grid;
  *b = call.block;
  *sh = call.sh;
  *st = call.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t sh, hipStream_t) {
  Launch l;
  l.k = &kernels.at(fn);
  if (!g.x || !g.y || !g.z || !b.x || b.x > 1024 || sh > max_lds) {
    bad.push_back(l.k->name + ": launch shape");
    return hipErrorInvalidValue;
  }
  for (size_t i = 0; i < l.k->args.size(); i++) {
    const std::string &t = l.k->args[i];
    l.ptr.push_back(t.back() == '*' ? *(const void **)args[i] : nullptr);
    if (t == "tmrx::SegPlan") {
      const tmrx::SegPlan &p = *(const tmrx::SegPlan *)args[i];
      l.plan.insert(l.plan.end(), {p.blk_lo, p.blk_seg, p.seg_blk, p.seg_tile});
    }
  }
  if (capture)
    capture->push_back(l);
  else
    run(l);
  return hipSuccess;
}
}
