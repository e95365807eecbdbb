// host_hip.cpp -- a stand-in for the HIP runtime on host memory, for tests of libqcu.so's
// host side without a GPU (allocation, error and bookkeeping paths).
//
// Loaded with global symbols before libqcu.so, its functions are the ones the library
// calls.  Device memory is host memory, an allocation can be made to fail, and kernels do
// not run: a launch is logged, and for the kernels below the model keeps which allocations
// hold links or clover blocks that some kernel has written, so that a launch which reads
// one that nothing has written is found.  As in HIP 7, a call that fails leaves its code
// for hipGetLastError and a later success does not clear it.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Alloc {
  size_t n;
  bool written;  // links or clover blocks, since it was allocated or the gauge last changed
};
std::map<const void*, std::string> g_names;
std::map<const void*, Alloc> g_mem;
std::vector<std::string> g_log;
std::map<std::string, double> g_cost;
std::map<hipEvent_t, double> g_events;
std::map<const void*, void*> g_symbols;
std::string g_wrong;
hipError_t g_last = hipSuccess;
long g_until_fail = -1;  // allocations until the one that fails, -1: none does
size_t g_live = 0;
long g_pinned = 0;
double g_clock = 0.0;
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_stream;

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}

void wrote(const void* p) {
  auto it = g_mem.find(p);
  if (it != g_mem.end()) it->second.written = true;
}
void reads(const std::string& kernel, const void* p) {
  auto it = g_mem.find(p);
  if (it == g_mem.end() || it->second.written) return;
  if (g_wrong.empty()) g_wrong = kernel + " reads " + std::to_string(it->second.n) + " bytes that nothing wrote";
}
bool is(const std::string& k, const char* part) { return k.find(part) != std::string::npos; }

uint64_t word_sum(const void* p, long words) {
  uint64_t s = 0;
  for (long i = 0; i < words; ++i) s += static_cast<const uint64_t*>(p)[i] * (uint64_t)(2 * i + 1);
  return s;
}

// what the model needs to know of a launch; a[i] points at argument i
void model(const std::string& k, void** a) {
  auto ptr = [&](int i) { return *static_cast<void**>(a[i]); };
  auto num = [&](int i) { return *static_cast<long*>(a[i]); };
  if (is(k, "clover_build_kernel")) {  // CloverBuild: links, A[2], A^-1[2]
    void* const* w = static_cast<void* const*>(a[0]);
    reads(k, w[0]);
    for (int i = 1; i < 5; ++i) wrote(w[i]);
  } else if (is(k, "clover_convert_kernel")) {
    reads(k, ptr(0));
    wrote(ptr(1));
  } else if (is(k, "clover_unpack_kernel") || is(k, "clover_apply_kernel")) {
    reads(k, ptr(0));
  } else if (is(k, "gauge_pack_kernelILi0ELi12ELi1E")) {  // import: every older field is of other links
    for (auto& m : g_mem) m.second.written = false;
    wrote(ptr(1));
    static_cast<uint64_t*>(ptr(3))[0] = word_sum(ptr(0), 8 * num(2) * 18);
  } else if (is(k, "gauge_pack_kernel")) {
    wrote(ptr(1));
  } else if (is(k, "gauge_repack_kernel")) {
    reads(k, ptr(0));
    wrote(ptr(1));
  } else if (is(k, "fingerprint_kernel")) {
    static_cast<uint64_t*>(ptr(2))[0] = word_sum(ptr(0), num(1) * 18);
  } else if (is(k, "hop_iface_kernel")) {  // IfaceArgs: links, clover by parity
    void* const* w = static_cast<void* const*>(a[0]);
    for (int i = 0; i < 3; ++i) reads(k, w[i]);
  } else if (is(k, "hop_split_kernel") || is(k, "hop_lds_kernel") || is(k, "10hop_kernel")) {
    void* const* w = static_cast<void* const*>(a[0]);  // HopArgs: in, out, x, links, 3 strides, clover[16]
    reads(k, w[3]);
    for (int i = 7; i < 23; ++i) reads(k, w[i]);
  }
}

}  // namespace

extern "C" {

// ------------------------------------------------------------ for the tests ---
// the n-th allocation from now fails (-1: none); returns how many were left until the last
// one that was asked for, -1 when it has failed
long host_hip_fail_after(long n) {
  const long left = g_until_fail;
  g_until_fail = n;
  return left;
}
size_t host_hip_live() { return g_live; }
long host_hip_pinned() { return g_pinned; }  // live pinned allocations
void host_hip_clear_log() {
  g_log.clear();
  g_wrong.clear();
}
long host_hip_launches(const char* part) {
  long n = 0;
  for (const std::string& k : g_log) n += is(k, part);
  return n;
}
// place of the first launch of such a kernel in the log, or -1
long host_hip_first(const char* part) {
  for (size_t i = 0; i < g_log.size(); ++i)
    if (is(g_log[i], part)) return (long)i;
  return -1;
}
const char* host_hip_wrong() { return g_wrong.c_str(); }
// the time, in ms, of a launch of kernels whose name has `part` (1 ms otherwise)
void host_hip_cost(const char* part, double ms) { g_cost[part] = ms; }

// ---------------------------------------------------------------- the runtime ---
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) {
  g_symbols[var] = calloc(1, size);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  g_grid = g;
  g_block = b;
  g_shmem = sh;
  g_stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st) {
  *g = g_grid;
  *b = g_block;
  *sh = g_shmem;
  *st = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3 block, void** args, size_t, hipStream_t) {
  const std::string k = g_names[f] + "/" + std::to_string(block.x);  // with its threads per block
  g_log.push_back(k);
  double ms = 1.0;
  for (auto& c : g_cost)
    if (is(k, c.first.c_str())) ms = c.second;
  g_clock += ms;
  model(k, args);
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (g_until_fail == 0) {
    g_until_fail = -1;
    return ret(hipErrorOutOfMemory);
  }
  if (g_until_fail > 0) --g_until_fail;
  if (n > (size_t)1 << 40) return ret(hipErrorOutOfMemory);
  *p = calloc(1, n);
  g_mem[*p] = {n, false};
  g_live += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = g_mem.find(p);
  if (it == g_mem.end()) return p ? ret(hipErrorInvalidValue) : hipSuccess;
  g_live -= it->second.n;
  g_mem.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n);
  ++g_pinned;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  if (p) --g_pinned;
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  wrote(d);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)1 << 33;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) {
  *p = g_symbols[sym];
  return hipSuccess;
}

hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }

hipError_t hipStreamCreate(hipStream_t* s) {
  *s = reinterpret_cast<hipStream_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  free(s);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) {
  free(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  free(e);
  return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  g_events.erase(e);
  free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  g_events[e] = g_clock;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(g_events[b] - g_events[a]);
  return hipSuccess;
}

}  // extern "C"
