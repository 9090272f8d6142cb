// A host-memory stand-in for the HIP calls the engine makes, loaded with RTLD_GLOBAL before
// libtotem.so so that the library's host code runs on a machine without a GPU.  Kernels do
// nothing.  Copies to the host are deferred until their stream is waited for, as copies into
// page-locked memory are; a test can limit the device's memory, make a copy fail, fill a
// copy of a given size with a value, and read what was allocated, launched and left pending.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace {
struct Copy {
  void* dst;
  const void* src;
  size_t bytes;
};
std::mutex mu;
std::map<void*, size_t> allocs;
std::map<hipStream_t, std::vector<Copy>> pending;
size_t capacity = (size_t)288 << 30, in_use = 0, peak = 0, in_use_at_info = 0;
size_t fill_bytes = 0;
int fill_value = 0;
long copies_to_fail = -1;      // copies to the host until one fails
long launches = 0, events = 0;
unsigned long long widest = 0;  // threads of the widest launch along x
hipError_t last = hipSuccess;
std::map<const void*, void*> symbols;

hipError_t fail(hipError_t e) {
  last = e;
  return e;
}
void drain(hipStream_t s) {
  for (const Copy& c : pending[s]) std::memcpy(c.dst, c.src, c.bytes);
  pending[s].clear();
}
void drain_all() {
  for (auto& p : pending) drain(p.first);
}
template <class T> T* handle() { return reinterpret_cast<T*>(std::malloc(1)); }
}  // namespace

extern "C" {

// ---------------------------------------------------------------- what a test sets and reads
void stub_capacity(size_t bytes) { capacity = bytes; }
void stub_fail_copy(long n) { copies_to_fail = n; }
void stub_fill(size_t bytes, int value) {
  fill_bytes = bytes;
  fill_value = value;
}
size_t stub_in_use() { return in_use; }
size_t stub_peak() { return peak; }
void stub_reset_peak() { peak = in_use; }
size_t stub_in_use_at_info() { return in_use_at_info; }
long stub_launches() { return launches; }
long stub_events() { return events; }
unsigned long long stub_widest() { return widest; }
long stub_pending() {
  long n = 0;
  for (auto& p : pending) n += (long)p.second.size();
  return n;
}

// ---------------------------------------------------------------------------- device, memory
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() {
  std::lock_guard<std::mutex> lk(mu);
  drain_all();
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* fr, size_t* total) {
  std::lock_guard<std::mutex> lk(mu);
  in_use_at_info = in_use;
  *fr = capacity - in_use;
  *total = capacity;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  if (bytes > capacity - in_use) return fail(hipErrorOutOfMemory);
  void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED) return fail(hipErrorOutOfMemory);
  allocs[m] = bytes;
  in_use += bytes;
  peak = std::max(peak, in_use);
  *p = m;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  drain_all();
  auto it = allocs.find(p);
  if (it == allocs.end()) return p ? fail(hipErrorInvalidValue) : hipSuccess;
  munmap(p, it->second);
  in_use -= it->second;
  allocs.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  if (kind != hipMemcpyDeviceToHost) {
    std::memcpy(dst, src, bytes);
    return hipSuccess;
  }
  if (copies_to_fail >= 0 && copies_to_fail-- == 0) return fail(hipErrorUnknown);
  if (fill_bytes && bytes == fill_bytes)
    for (size_t i = 0; i < bytes / sizeof(int); ++i) reinterpret_cast<int*>(const_cast<void*>(src))[i] = fill_value;
  pending[s].push_back({dst, src, bytes});
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) {
  std::lock_guard<std::mutex> lk(mu);
  void*& m = symbols[sym];
  if (!m) m = mmap(nullptr, (size_t)256 << 20, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  *p = m;
  return hipSuccess;
}

// ------------------------------------------------------------------- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(handle<char>());
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  drain(s);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(handle<char>());
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(handle<char>());
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  ++events;
  *e = reinterpret_cast<hipEvent_t>(handle<char>());
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipDeviceSynchronize(); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}

// ------------------------------------------------------------------------- kernels, errors
struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
static thread_local Config config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
  config = {grid, block, shared, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  ++launches;
  const unsigned long long x = (unsigned long long)grid.x * block.x;
  widest = std::max(widest, x);
  // threads of a launch along one dimension are counted in 32 bits
  if (grid.x == 0 || x > 0xffffffffull) return fail(hipErrorInvalidConfiguration);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }

}  // extern "C"
