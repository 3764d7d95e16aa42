// The HIP runtime calls libgpufem makes, over host memory and without a GPU:
// device memory is calloc'ed, kernels are recorded by name instead of run
// (except the ELL expansion, which the host code reads back), and the test
// decides which allocation or launch fails, how much memory there is and how
// long a kernel takes.  Errors stay until hipGetLastError reads them, as in
// HIP 7.  Loaded with global visibility before libgpufem.so.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <unordered_map>
#include <vector>

namespace {

struct Fake {
  std::unordered_map<void*, size_t> mem;
  size_t live_bytes = 0, total_bytes = size_t(8) << 30, largest = ~size_t(0);
  int64_t mallocs = 0, fail_at = -1, h2d = 0, last_bytes = 0;
  hipError_t last = hipSuccess;
  double clock_ms = 0.0;
  std::map<std::string, double> cost_us;  // by part of the name; else 1
  std::string stop;                       // a launch whose name contains it fails
  std::string log;
  std::unordered_map<const void*, std::string> names;
  dim3 grid, block;
  size_t shared = 0;
  hipStream_t stream = nullptr;
};
Fake& F() {
  static Fake* f = new Fake();
  return *f;
}
hipError_t err(hipError_t e) {
  if (e != hipSuccess) F().last = e;
  return e;
}

// (n, width, dim, adj_ptr, adj, val, col, rownnz)
void ell_expand(void** a) {
  const int64_t n = *static_cast<int64_t*>(a[0]);
  const int32_t width = *static_cast<int32_t*>(a[1]), dim = *static_cast<int*>(a[2]);
  const int64_t* ptr = *static_cast<const int64_t**>(a[3]);
  const int32_t* adj = *static_cast<const int32_t**>(a[4]);
  int32_t* col = *static_cast<int32_t**>(a[6]);
  int32_t* rownnz = *static_cast<int32_t**>(a[7]);
  for (int64_t row = 0; row < n; ++row) {
    const int64_t v = row / dim;
    rownnz[row] = int32_t(ptr[v + 1] - ptr[v]) * dim;
    for (int32_t s = 0; s < width; ++s)
      col[row + s * n] = s < rownnz[row] ? adj[ptr[v] + s / dim] * dim + s % dim : int32_t(row);
  }
}

hipError_t launch(const void* f, void** args) {
  const std::string& name = F().names[f];
  F().log += name + "\n";
  if (!F().stop.empty() && name.find(F().stop) != std::string::npos) return err(hipErrorLaunchFailure);
  double us = 1.0;
  for (const auto& c : F().cost_us)
    if (name.find(c.first) != std::string::npos) us = c.second;
  F().clock_ms += 1e-3 * us;
  if (name.find("k_ell_expand") != std::string::npos) ell_expand(args);
  return hipSuccess;
}

}  // namespace

extern "C" {

// ---- the test's side -------------------------------------------------------------
void fake_fail_at(int64_t k) { F().fail_at = k < 0 ? -1 : F().mallocs + k; }  // k-th from now
void fake_memory(int64_t total, int64_t largest) {
  F().total_bytes = size_t(total);
  F().largest = largest > 0 ? size_t(largest) : ~size_t(0);
}
void fake_stop(const char* name) { F().stop = name; }
void fake_cost(const char* name, double us) { F().cost_us[name] = us; }
int64_t fake_live() { return int64_t(F().mem.size()); }
int64_t fake_live_bytes() { return int64_t(F().live_bytes); }
int64_t fake_mallocs() { return F().mallocs; }
int64_t fake_h2d() { return F().h2d; }
int64_t fake_last_bytes() { return F().last_bytes; }  // of the last allocation asked for
const char* fake_log() { return F().log.c_str(); }
void fake_clear_log() { F().log.clear(); }

// ---- the library's side ----------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*,
                           uint3*, dim3*, dim3*, int*) {
  F().names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
  F().grid = g, F().block = b, F().shared = shared, F().stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* s) {
  *g = F().grid, *b = F().block, *shared = F().shared, *s = F().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  return launch(f, args);
}
hipError_t hipLaunchCooperativeKernel(const void* f, dim3, dim3, void** args, unsigned, hipStream_t) {
  return launch(f, args);
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 3;
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  const int64_t k = F().mallocs++;
  F().last_bytes = int64_t(bytes);
  if (k == F().fail_at || bytes > F().largest || F().live_bytes + bytes > F().total_bytes)
    return err(hipErrorOutOfMemory);
  *p = std::calloc(bytes > 0 ? bytes : 1, 1);
  F().mem[*p] = bytes;
  F().live_bytes += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  auto it = F().mem.find(p);
  if (it == F().mem.end()) return err(hipErrorInvalidValue);
  F().live_bytes -= it->second;
  F().mem.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total_b) {
  *total_b = F().total_bytes;
  *free_b = F().total_bytes - F().live_bytes;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind kind) {
  std::memcpy(d, s, n);
  if (kind == hipMemcpyHostToDevice) F().h2d += int64_t(n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
  return hipMemcpy(d, s, n, kind);
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) {
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* area = std::calloc(size_t(64) << 20, 1);
  *p = area;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->maxSharedMemoryPerMultiProcessor = 160 * 1024;
  std::strcpy(p->gcnArchName, "none");
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new int());
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete reinterpret_cast<int*>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(new int());
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return err(hipErrorLaunchFailure); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete reinterpret_cast<int*>(e);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(new double(0.0));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<double*>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  *reinterpret_cast<double*>(e) = F().clock_ms;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = float(*reinterpret_cast<double*>(b) - *reinterpret_cast<double*>(a));
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : e == hipSuccess ? "no error" : "error";
}
hipError_t hipGetLastError(void) {
  const hipError_t e = F().last;
  F().last = hipSuccess;
  return e;
}

}  // extern "C"
