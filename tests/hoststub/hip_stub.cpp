// hip_stub.cpp -- the HIP calls of the host library without a GPU, for the CPU
// tests of what it launches, copies and allocates (tests/test_host_launches.py).
//
// Memory is ordinary memory, copies are made at once, kernels do nothing.
// Every launch is logged by name; a force launch that also makes the advance
// and the next insert is logged as name+next, a launch inside a capture when
// its graph is launched.  Events carry a clock that each launch moves on (see
// cost), so that what the library measures is the same in every run.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <vector>

#include "fx_common.hpp"
#include "noalloc.hpp"

namespace {

struct Event {
  double at = 0.0;
};
struct Graph {
  std::vector<std::string> launches;
};

std::string g_log;
std::vector<std::string>* g_capture = nullptr;
std::map<std::string, void*> g_functions, g_globals;
double g_clock = 0.0;
long g_launches = 0, g_captures = 0, g_events = 0, g_waits = 0;
size_t g_pinned = 0;
bool g_no_pinned = false;
std::map<void*, size_t> g_pin;
thread_local long g_fail_new = 0;  // the call of operator new, from now, that throws

struct Own {  // memory that a stub takes for itself does not count
  const long armed = g_fail_new;
  Own() { g_fail_new = 0; }
  ~Own() { g_fail_new = armed; }
};

const char* name_of(hipFunction_t f) {
  for (const auto& e : g_functions)
    if (e.second == (void*)f) return e.first.c_str();
  return "?";
}

// Fewer blocks are faster, and every launch a little faster than the one
// before: what is tried last looks best where nothing else differs.  A force
// that also advances and inserts is fastest in small blocks.
double cost(const std::string& k, unsigned blocks, unsigned threads) {
  const double drift = 1.0 - 1e-7 * (double)g_launches;
  if (k.find("+next") != std::string::npos) return (1.0 + 1e-3 * threads) * drift;
  return (1.0 + 1e-3 * blocks) * drift;
}

}  // namespace

void* operator new(size_t n) {
  if (g_fail_new > 0 && --g_fail_new == 0) throw std::bad_alloc();
  void* p = malloc(n ? n : 1);
  if (p == nullptr) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

int fx::scratch_setup(void** out) {
  static uint32_t words[FX_SCAN_SCRATCH_WORDS];
  *out = words;
  return FX_OK;
}

extern "C" {

// what the tests read and set
const char* stub_log() { return g_log.c_str(); }
void stub_clear_log() { g_log.clear(); }
long stub_captures() { return g_captures; }
long stub_events() { return g_events; }
long stub_waits() { return g_waits; }  // for a stream
long stub_pinned_bytes() { return (long)g_pinned; }
void stub_fail_new(long nth) { g_fail_new = nth; }
void stub_no_pinned(int on) { g_no_pinned = on != 0; }
hipError_t hipGetLastError() { return hipSuccess; }

const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)1 << 30;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_no_pinned) return hipErrorOutOfMemory;
  const Own own;
  const hipError_t e = hipMalloc(p, n);
  if (e == hipSuccess) {
    g_pin[*p] = n;
    g_pinned += n;
  }
  return e;
}
hipError_t hipHostFree(void* p) {
  g_pinned -= g_pin[p];
  g_pin.erase(p);
  return hipFree(p);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpyDtoH(void* d, hipDeviceptr_t s, size_t n) { return hipMemcpy(d, s, n, hipMemcpyDeviceToHost); }
hipError_t hipMemcpyHtoD(hipDeviceptr_t d, const void* s, size_t n) { return hipMemcpy(d, s, n, hipMemcpyHostToDevice); }
hipError_t hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t* e) {
  const Own own;
  g_events++;
  *e = (hipEvent_t) new Event;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  ((Event*)e)->at = g_clock;
  return hipSuccess;
}
hipError_t hipEventRecordWithFlags(hipEvent_t e, hipStream_t s, unsigned) { return hipEventRecord(e, s); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(((Event*)b)->at - ((Event*)a)->at);
  return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t)malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  free((void*)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  g_waits++;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_captures++;
  g_capture = &(new Graph)->launches;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)g_capture;
  g_capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t) new Graph{*(std::vector<std::string>*)g};
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
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (const std::string& k : ((Graph*)e)->launches) g_log += k + "\n";
  return hipSuccess;
}

hipError_t hipModuleLoad(hipModule_t* m, const char*) {
  *m = (hipModule_t)malloc(1);
  return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t m) {
  free((void*)m);
  return hipSuccess;
}
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* k) {
  void*& p = g_functions[k];
  if (p == nullptr) p = malloc(1);
  *f = (hipFunction_t)p;
  return hipSuccess;
}
hipError_t hipModuleGetGlobal(hipDeviceptr_t* p, size_t* n, hipModule_t, const char* k) {
  const std::map<std::string, size_t> size = {{"FParams", sizeof(FParams_t)}, {"FPnts", sizeof(cuDataX)},
                                              {"FPntTmp", sizeof(cuDataX)},   {"FAccel", sizeof(cuDataX)},
                                              {"FNbrWords", sizeof(int)},     {"FSortSrc", sizeof(void*)},
                                              {"FHostCaps", sizeof(int)},     {"FPpt", 8 * sizeof(int)}};
  const auto it = size.find(k);
  if (it == size.end()) return hipErrorNotFound;
  void*& g = g_globals[k];
  if (g == nullptr) g = calloc(1, it->second);
  *p = (hipDeviceptr_t)g;
  *n = it->second;
  return hipSuccess;
}
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned bx, unsigned, unsigned, unsigned tx, unsigned, unsigned,
                                 unsigned, hipStream_t, void** args, void**) {
  std::string k = name_of(f);
  if (k.find("computeForceWave") == 0) {  // its last argument begins with what follows the forces
    const int at = k.find("Batch") == std::string::npos ? 3 : 4;
    if (*(const int*)args[at] != 0) k += "+next";
  }
  g_launches++;
  g_clock += cost(k, bx, tx);
  if (g_capture != nullptr)
    g_capture->push_back(k);
  else
    g_log += k + "\n";
  return hipSuccess;
}

}  // extern "C"
