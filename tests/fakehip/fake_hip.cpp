// A HIP runtime without a device, for CPU tests of the library's host paths:
// device memory is host memory, kernels do nothing, and every call that orders
// work goes to a log that the test reads.  Loaded before libsrg_tdbp.so, so the
// library's HIP calls resolve here (tests/fakehip/__init__.py).
#include <hip/hip_runtime_api.h>

#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::condition_variable cv;
std::map<const void*, std::string> kernels;   // host stub -> mangled device name
std::vector<std::string> calls;
std::map<std::string, int> fail_in;           // call -> how many more succeed
std::set<void*> blocked;                      // streams that hipStreamSynchronize waits on
std::map<void*, int> waiting;
std::map<const void*, int> owner;             // pointers said to be another device's
std::map<void*, std::vector<std::string>> capture, graphs;   // stream / graph -> launches
std::map<void*, double> clock_of, stamp;      // simulated ms of a stream, of an event
struct Cost {
  std::string part;   // of a kernel's name
  double alone, among;   // ms, in a graph that holds no other such kernel, or others
};
std::vector<Cost> costs;
thread_local hipError_t last = hipSuccess;
thread_local int device = 0;
int devices = 1;
struct Launch {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local std::vector<Launch> config;

std::string hex(const void* p) {
  char b[32];
  snprintf(b, sizeof b, "%p", p ? p : (const void*)0x1);
  return b;
}
hipError_t note(const char* call, const std::string& text = "") {
  std::lock_guard<std::mutex> lk(mu);
  auto it = fail_in.find(call);
  if (it != fail_in.end() && it->second-- <= 0) {
    fail_in.erase(it);
    return last = hipErrorUnknown;
  }
  if (!text.empty()) calls.push_back(std::string(call) + " " + text);
  return hipSuccess;
}
const Cost* cost(const std::string& name) {
  for (auto& c : costs)
    if (name.find(c.part) != std::string::npos) return &c;
  return nullptr;
}
}  // namespace

extern "C" {

// ---- the test's side
int fake_log(char* out, int n) {
  std::lock_guard<std::mutex> lk(mu);
  std::string all;
  for (auto& c : calls) all += c + "\n";
  if ((int)all.size() < n) std::memcpy(out, all.c_str(), all.size() + 1);
  return (int)all.size() + 1;
}
void fake_clear() {
  std::lock_guard<std::mutex> lk(mu);
  calls.clear();
}
void fake_fail(const char* call, int after) {
  std::lock_guard<std::mutex> lk(mu);
  fail_in[call] = after;
}
void fake_block(void* s, int on) {
  std::lock_guard<std::mutex> lk(mu);
  if (on) blocked.insert(s);
  else blocked.erase(s);
  cv.notify_all();
}
int fake_waiting(void* s) {
  std::lock_guard<std::mutex> lk(mu);
  return waiting[s];
}
void fake_owner(void* p, int dev) {
  std::lock_guard<std::mutex> lk(mu);
  owner[p] = dev;
}
void fake_cost(const char* part, double alone, double among) {
  std::lock_guard<std::mutex> lk(mu);
  costs.insert(costs.begin(), {part, alone, among});
}

// ---- kernels
void** __hipRegisterFatBinary(const void*) { return (void**)std::calloc(1, 8); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           dim3*, dim3*, int*) {
  std::lock_guard<std::mutex> lk(mu);
  kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  config.push_back({g, b, m, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  const Launch l = config.back();
  config.pop_back();
  *g = l.grid;
  *b = l.block;
  *m = l.shared;
  *s = l.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t s) {
  std::string name;
  {
    std::lock_guard<std::mutex> lk(mu);
    name = kernels[f];
    auto c = capture.find(s);
    if (c != capture.end()) {
      c->second.push_back(name);
      return hipSuccess;
    }
    if (const Cost* k = cost(name)) clock_of[s] += k->alone;
  }
  return note("hipLaunchKernel", hex(s) + " " + name);
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e ? "fake error" : "no error"; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* scratch = std::calloc(1, 1 << 20);
  *p = scratch;
  return hipSuccess;
}

// ---- devices
hipError_t hipGetDeviceCount(int* n) {
  *n = devices;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  device = d;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)1 << 38;
  return hipSuccess;
}

// ---- memory
hipError_t hipMalloc(void** p, size_t n) {
  if (note("hipMalloc")) return hipErrorOutOfMemory;
  *p = std::calloc(n, 1);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  note("hipFree", hex(p));
  return hipSuccess;   // kept: the log names memory by its address
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void*, hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (note("hipHostMalloc", std::to_string(n))) return hipErrorOutOfMemory;
  *p = std::calloc(n, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  note("hipHostFree", hex(p));
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::lock_guard<std::mutex> lk(mu);
  std::memset(a, 0, sizeof *a);
  a->type = hipMemoryTypeDevice;
  auto it = owner.find(p);
  a->device = it == owner.end() ? device : it->second;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  if (note("hipMemcpyAsync", hex(st) + " " + hex(d) + " " + hex(s))) return last;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t st) {
  if (note("hipMemcpy2DAsync", hex(st))) return last;
  for (size_t i = 0; i < h; ++i) std::memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)std::calloc(1, 8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::unique_lock<std::mutex> lk(mu);
  if (capture.count(s)) return last = hipErrorStreamCaptureUnsupported;
  ++waiting[s];
  cv.notify_all();
  cv.wait(lk, [&] { return !blocked.count(s); });
  --waiting[s];
  calls.push_back("hipStreamSynchronize " + hex(s));
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return note("hipDeviceSynchronize", "-"); }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)std::calloc(1, 8);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  {
    std::lock_guard<std::mutex> lk(mu);
    stamp[e] = clock_of[s];
  }
  return note("hipEventRecord", hex(s) + " " + hex(e));
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  return note("hipStreamWaitEvent", hex(s) + " " + hex(e));
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  std::lock_guard<std::mutex> lk(mu);
  *ms = (float)(stamp[b] - stamp[a]);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  std::lock_guard<std::mutex> lk(mu);
  *st = capture.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  std::lock_guard<std::mutex> lk(mu);
  capture[s];
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  std::lock_guard<std::mutex> lk(mu);
  *g = (hipGraph_t)std::calloc(1, 8);
  graphs[*g] = capture[s];
  capture.erase(s);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)g;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  int timed = 0;
  for (auto& name : graphs[e]) timed += cost(name) && cost(name)->alone > 0;
  for (auto& name : graphs[e]) {
    if (const Cost* k = cost(name)) clock_of[s] += timed > 1 ? k->among : k->alone;
    calls.push_back("hipLaunchKernel " + hex(s) + " " + name);
  }
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

// ---- rocFFT: a transform is a launch on its plan's stream
int rocfft_setup() { return 0; }
int rocfft_plan_create(void** p, int, int, int, size_t, const size_t*, size_t, void*) {
  *p = std::calloc(1, 8);
  return 0;
}
int rocfft_plan_destroy(void*) { return 0; }
int rocfft_plan_get_work_buffer_size(void*, size_t* n) {
  *n = 0;
  return 0;
}
int rocfft_execution_info_create(void** i) {
  *i = std::calloc(1, 8);
  return 0;
}
int rocfft_execution_info_destroy(void*) { return 0; }
int rocfft_execution_info_set_stream(void* i, void* s) {
  *(void**)i = s;
  return 0;
}
int rocfft_execution_info_set_work_buffer(void*, void*, size_t) { return 0; }
int rocfft_execute(void*, void**, void**, void* i) {
  return note("hipLaunchKernel", hex(*(void**)i) + " rocfft");
}

}  // extern "C"
