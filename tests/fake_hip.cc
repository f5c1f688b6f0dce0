/* The part of the HIP runtime that libkifmm.so calls, on the host: device
 * memory is host memory, a kernel launch does nothing but appear in a log and
 * advance a clock, and calls can be made to fail.  What the library's host code
 * does with the runtime (what it takes, gives back, launches, waits for and
 * times, and what it makes of an error) is then tested without a GPU
 * (tests/fake_device.py).  Loaded before the library, so that its names are
 * found first.  A use of memory, a stream or an event that is not live is
 * kept in a list of faults. */
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace {

struct Fake {
  std::recursive_mutex m;
  struct Mem {
    size_t bytes;
    unsigned id;
  };
  std::map<char*, Mem> dev, pin;                /* live allocations */
  std::vector<void*> dead;                      /* freed ones, kept mapped so that a stray access is a fault entry, not a crash */
  struct Stream {
    int id;
    bool capturing;
  };
  std::map<hipStream_t, Stream> streams;        /* live ones */
  std::map<hipEvent_t, double> events;          /* live; time recorded, < 0: none */
  std::map<const void*, std::string> kernels, vars;
  std::map<const void*, size_t> var_bytes;
  std::map<const void*, void*> var_mem;
  struct Fail {
    long skip, count;
    hipError_t e;
  };
  std::map<std::string, Fail> fails;
  std::map<std::string, long> calls;
  std::vector<std::pair<std::string, double>> cost; /* part of a kernel's name, ms */
  std::string log, faults;
  hipError_t last = hipSuccess;
  double clock = 0.0;
  size_t limit = (size_t)1 << 40, used = 0;
  unsigned next_id = 1;
  int next_stream = 0;
  struct {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
  } conf;
};
Fake& F() {
  static Fake* f = new Fake;
  return *f;
}
typedef std::lock_guard<std::recursive_mutex> Lock;

hipError_t done(hipError_t e) {
  if (e != hipSuccess) F().last = e; /* stays until it is read */
  return e;
}
/* whether this call of fn was asked to fail */
hipError_t asked(const char* fn) {
  F().calls[fn]++;
  auto it = F().fails.find(fn);
  if (it == F().fails.end() || it->second.count == 0) return hipSuccess;
  if (it->second.skip-- > 0) return hipSuccess;
  it->second.skip = 0;
  it->second.count--;
  return done(it->second.e);
}
#define ENTER(fn)                                                  \
  Lock lock(F().m);                                                \
  if (const hipError_t asked_ = asked(fn); asked_ != hipSuccess) return asked_

hipError_t fault(const std::string& what) {
  F().faults += what + "\n";
  return done(hipErrorInvalidValue);
}
const std::pair<char* const, Fake::Mem>* find(const std::map<char*, Fake::Mem>& m, const void* p, size_t n) {
  auto it = m.upper_bound((char*)p);
  if (it == m.begin()) return nullptr;
  --it;
  return (char*)p + n <= it->first + it->second.bytes ? &*it : nullptr;
}
bool live(const void* p, size_t n) { return find(F().dev, p, n) || find(F().pin, p, n); }
bool stream_ok(hipStream_t s, const char* fn) {
  if (!s || F().streams.count(s)) return true;
  F().faults += std::string(fn) + " on a stream that is not live\n";
  return false;
}
std::string id(hipStream_t s) { return s ? std::to_string(F().streams[s].id) : "null"; }
hipError_t alloc(std::map<char*, Fake::Mem>& m, void** p, size_t n) {
  char* const q = (char*)std::calloc(1, n ? n : 1);
  if (!q) return done(hipErrorOutOfMemory);
  m[q] = {n, F().next_id++};
  *p = q;
  return hipSuccess;
}
hipError_t launch(const char* fn, const void* f, dim3 g, dim3 b, hipStream_t s, hipEvent_t start, hipEvent_t stop) {
  if (!stream_ok(s, fn)) return hipErrorInvalidValue;
  auto it = F().kernels.find(f);
  const std::string name = it == F().kernels.end() ? "?" : it->second;
  double ms = 1.0;
  for (auto& c : F().cost)
    if (name.find(c.first) != std::string::npos) ms = c.second;
  if (start) F().events[start] = F().clock;
  F().clock += ms;
  if (stop) F().events[stop] = F().clock;
  F().log += "kernel " + id(s) + " " + std::to_string(g.x) + "x" + std::to_string(g.y) + "x" + std::to_string(g.z) + " " +
             std::to_string(b.x) + " " + name + "\n";
  return hipSuccess;
}
hipError_t copy(const char* fn, void* d, const void* s, size_t n, hipMemcpyKind k, const std::string& on) {
  const bool to_dev = k == hipMemcpyHostToDevice || k == hipMemcpyDeviceToDevice;
  const bool from_dev = k == hipMemcpyDeviceToHost || k == hipMemcpyDeviceToDevice;
  if ((to_dev && !live(d, n)) || (from_dev && !live(s, n))) return fault(std::string(fn) + " of memory that is not live");
  std::memcpy(d, s, n);
  F().log += std::string("copy ") + on + " " + (k == hipMemcpyHostToDevice ? "h2d " : k == hipMemcpyDeviceToHost ? "d2h " : "d2d ") +
             std::to_string(n) + "\n";
  return hipSuccess;
}

}  // namespace

extern "C" {

/* ---- what a test calls */
void fake_fail(const char* fn, long skip, long count, int e) {
  Lock lock(F().m);
  F().fails[fn] = {skip, count, (hipError_t)e};
}
long fake_calls(const char* fn) { return F().calls[fn]; }
void fake_kernel_ms(const char* part, double ms) { F().cost.emplace_back(part, ms); }
void fake_limit(size_t bytes) { F().limit = bytes; }
size_t fake_used() { return F().used; }
long fake_streams() { return (long)F().streams.size(); }
long fake_events() { return (long)F().events.size(); }
const char* fake_log() { return F().log.c_str(); }
void fake_clear_log() { F().log.clear(); }
const char* fake_faults() { return F().faults.c_str(); }
/* hipDeviceReset: nothing of the device lives on */
void fake_reset() {
  Lock lock(F().m);
  for (auto* m : {&F().dev, &F().pin}) {
    for (auto& p : *m) F().dead.push_back(p.first);
    m->clear();
  }
  for (auto& v : F().var_mem) F().pin[(char*)v.second] = {F().var_bytes[v.first], 0}; /* the program's own variables stay */
  F().used = 0;
  F().streams.clear();
  F().events.clear();
}

/* ---- the runtime */
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  int st = 0;
  char* const d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  F().kernels[f] = d ? d : name;
  std::free(d);
}
void __hipRegisterVar(void**, void* var, char*, char* name, int, size_t size, int, int) {
  F().vars[var] = name;
  F().var_bytes[var] = size;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  F().m.lock();
  F().conf = {g, b, sh, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
  *g = F().conf.grid, *b = F().conf.block, *sh = F().conf.shmem, *s = F().conf.stream;
  F().m.unlock();
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s) {
  ENTER("hipLaunchKernel");
  return launch("hipLaunchKernel", f, g, b, s, nullptr, nullptr);
}
hipError_t hipExtLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s, hipEvent_t start,
                              hipEvent_t stop, int) {
  ENTER("hipExtLaunchKernel");
  return launch("hipExtLaunchKernel", f, g, b, s, start, stop);
}
hipError_t hipMalloc(void** p, size_t n) {
  ENTER("hipMalloc");
  if (F().used + n > F().limit) return done(hipErrorOutOfMemory);
  F().used += n;
  return alloc(F().dev, p, n);
}
hipError_t hipFree(void* p) {
  ENTER("hipFree");
  if (!p) return hipSuccess;
  auto it = F().dev.find((char*)p);
  if (it == F().dev.end()) return fault("hipFree of memory that is not live");
  F().used -= it->second.bytes;
  F().dead.push_back(p);
  F().dev.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ENTER("hipHostMalloc");
  return alloc(F().pin, p, n);
}
hipError_t hipHostFree(void* p) {
  ENTER("hipHostFree");
  if (!p) return hipSuccess;
  if (!F().pin.count((char*)p)) return fault("hipHostFree of memory that is not live");
  F().dead.push_back(p);
  F().pin.erase((char*)p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  ENTER("hipHostGetDevicePointer");
  *d = h;
  return hipSuccess;
}
hipError_t hipPointerGetAttribute(void* out, hipPointer_attribute what, hipDeviceptr_t p) {
  ENTER("hipPointerGetAttribute");
  const auto* a = find(F().dev, p, 1);
  if (!a || what != HIP_POINTER_ATTRIBUTE_BUFFER_ID) return done(hipErrorInvalidValue);
  *(unsigned long long*)out = 0;
  std::memcpy(out, &a->second.id, sizeof(unsigned));
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  ENTER("hipMemcpy");
  return copy("hipMemcpy", d, s, n, k, "null");
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  ENTER("hipMemcpyAsync");
  if (!stream_ok(st, "hipMemcpyAsync")) return hipErrorInvalidValue;
  return copy("hipMemcpyAsync", d, s, n, k, id(st));
}
hipError_t hipMemset(void* d, int v, size_t n) {
  ENTER("hipMemset");
  if (!live(d, n)) return fault("hipMemset of memory that is not live");
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t s) {
  ENTER("hipMemsetAsync");
  if (!stream_ok(s, "hipMemsetAsync")) return hipErrorInvalidValue;
  return hipMemset(d, v, n);
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  ENTER("hipStreamCreate");
  *s = (hipStream_t)std::malloc(16);
  F().streams[*s] = {F().next_stream++, false};
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t s) {
  ENTER("hipStreamDestroy");
  if (!stream_ok(s, "hipStreamDestroy")) return hipErrorInvalidValue;
  F().streams.erase(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  ENTER("hipStreamSynchronize");
  return stream_ok(s, "hipStreamSynchronize") ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  ENTER("hipStreamWaitEvent");
  if (!stream_ok(s, "hipStreamWaitEvent")) return hipErrorInvalidValue;
  return F().events.count(e) ? hipSuccess : fault("hipStreamWaitEvent for an event that is not live");
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  ENTER("hipStreamBeginCapture");
  if (!stream_ok(s, "hipStreamBeginCapture")) return hipErrorInvalidValue;
  F().streams[s].capturing = true;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  ENTER("hipStreamEndCapture");
  if (!F().streams.count(s) || !F().streams[s].capturing) return fault("hipStreamEndCapture of a stream that does not capture");
  F().streams[s].capturing = false;
  *g = (hipGraph_t)std::malloc(16);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  ENTER("hipGraphInstantiate");
  *x = (hipGraphExec_t)std::malloc(16);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  ENTER("hipGraphLaunch");
  F().log += "graph " + id(s) + "\n";
  F().clock += 1.0;
  return stream_ok(s, "hipGraphLaunch") ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  ENTER("hipEventCreate");
  *e = (hipEvent_t)std::malloc(16);
  F().events[*e] = -1.0;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  ENTER("hipEventDestroy");
  return F().events.erase(e) ? hipSuccess : fault("hipEventDestroy of an event that is not live");
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  ENTER("hipEventRecord");
  if (!stream_ok(s, "hipEventRecord")) return hipErrorInvalidValue;
  if (!F().events.count(e)) return fault("hipEventRecord of an event that is not live");
  F().events[e] = F().clock;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  ENTER("hipEventSynchronize");
  return F().events.count(e) ? hipSuccess : fault("hipEventSynchronize of an event that is not live");
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  ENTER("hipEventElapsedTime");
  if (!F().events.count(a) || !F().events.count(b)) return fault("hipEventElapsedTime of an event that is not live");
  if (F().events[a] < 0.0 || F().events[b] < 0.0) return done(hipErrorInvalidHandle); /* not recorded */
  *ms = (float)(F().events[b] - F().events[a]);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
  ENTER("hipDeviceSynchronize");
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  ENTER("hipSetDevice");
  return d == 0 ? hipSuccess : done(hipErrorInvalidDevice);
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  Lock lock(F().m);
  const hipError_t e = F().last;
  F().last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  static thread_local char s[32];
  std::snprintf(s, sizeof s, "fake error %d", (int)e);
  return s;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) {
  ENTER("hipGetSymbolAddress");
  if (!F().var_bytes.count(sym)) return fault("hipGetSymbolAddress of an unknown symbol");
  void*& m = F().var_mem[sym];
  if (!m) {
    (void)alloc(F().pin, &m, F().var_bytes[sym]);
  }
  *p = m;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeWarpSize ? 64 : a == hipDeviceAttributeMultiprocessorCount ? 256 : 1024;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset((void*)p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->warpSize = 64;
  p->multiProcessorCount = 256;
  p->maxThreadsPerBlock = 1024;
  p->maxThreadsPerMultiProcessor = 2048;
  p->sharedMemPerBlock = 65536;
  p->maxGridSize[0] = 1 << 30;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }

}  // extern "C"
