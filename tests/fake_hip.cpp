// The HIP runtime calls that libheatgeo makes, for tests of its host code where there is no GPU:
// device memory is host memory (zeroed), a launch is a line in a log and runs nothing, a copy is a
// memcpy. Loaded with RTLD_GLOBAL before libheatgeo.so, whose calls then bind here. A test can make
// the n-th allocation from now fail, and hold the next thread that launches a kernel of some name
// until it opens the gate.
#include <hip/hip_runtime_api.h>

#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct State {
  std::mutex lock;
  std::condition_variable changed;
  std::map<const void*, std::string> names;  // a kernel's host stub -> its mangled name
  std::map<char*, size_t> live;              // device allocations
  std::vector<std::string> launched;
  long fail_in = 0;  // the allocation that fails, counted from 1; 0: none does
  std::string gate;
  int waiting = 0;
  bool open = false;
};

State& state() {  // libheatgeo's constructors register its kernels
  static State* s = new State;
  return *s;
}

thread_local std::vector<std::string> t_launched;
thread_local dim3 t_grid, t_block;
thread_local size_t t_shared;
thread_local hipStream_t t_stream;

hipError_t launch(const void* function) {
  State& s = state();
  std::unique_lock<std::mutex> hold(s.lock);
  const std::string& name = s.names[function];
  s.launched.push_back(name);
  t_launched.push_back(name);
  if (!s.gate.empty() && name.find(s.gate) != std::string::npos) {
    s.gate.clear();
    ++s.waiting;
    s.changed.notify_all();
    s.changed.wait(hold, [&] { return s.open; });
    --s.waiting;
  }
  return hipSuccess;
}

hipError_t allocate(void** out, size_t bytes) {
  State& s = state();
  std::lock_guard<std::mutex> hold(s.lock);
  if (s.fail_in > 0 && --s.fail_in == 0) {
    *out = nullptr;
    return hipErrorOutOfMemory;
  }
  *out = std::calloc(1, bytes > 0 ? bytes : 1);
  s.live[static_cast<char*>(*out)] = bytes;
  return hipSuccess;
}

long count(const std::vector<std::string>& log, const char* part) {
  long found = 0;
  for (const std::string& name : log) found += name.find(part) != std::string::npos;
  return found;
}

hipError_t copy(void* to, const void* from, size_t bytes) {
  if (bytes > 0 && (!to || !from)) return hipErrorInvalidValue;
  if (bytes > 0) std::memcpy(to, from, bytes);
  return hipSuccess;
}

int g_handle;  // what every stream, event and graph points at
template <typename T>
T handle() {
  return reinterpret_cast<T>(&g_handle);
}

}  // namespace

extern "C" {

// ---- the tests' side ----------------------------------------------------------------------------

void fake_fail_allocation(long n) {
  std::lock_guard<std::mutex> hold(state().lock);
  state().fail_in = n;
}
// Whether the allocation that was to fail is still to come (disarmed here).
int fake_failure_pending() {
  std::lock_guard<std::mutex> hold(state().lock);
  const bool pending = state().fail_in > 0;
  state().fail_in = 0;
  return pending;
}
long fake_live_bytes() {
  std::lock_guard<std::mutex> hold(state().lock);
  long total = 0;
  for (const auto& a : state().live) total += static_cast<long>(a.second);
  return total;
}
// Launches of kernels whose mangled names hold `part`: of the process, of the calling thread.
long fake_launches(const char* part) {
  std::lock_guard<std::mutex> hold(state().lock);
  return count(state().launched, part);
}
long fake_thread_launches(const char* part) { return count(t_launched, part); }
void fake_gate(const char* part) {
  std::lock_guard<std::mutex> hold(state().lock);
  state().gate = part;
  state().open = false;
}
// Waits (ten seconds at most) for a thread to stand at the gate.
int fake_held() {
  std::unique_lock<std::mutex> hold(state().lock);
  return state().changed.wait_for(hold, std::chrono::seconds(10), [] { return state().waiting > 0; });
}
void fake_open() {
  std::lock_guard<std::mutex> hold(state().lock);
  state().gate.clear();
  state().open = true;
  state().changed.notify_all();
}

// ---- the runtime's side -------------------------------------------------------------------------

void** __hipRegisterFatBinary(const void*) { return handle<void**>(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  std::lock_guard<std::mutex> hold(state().lock);
  state().names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  t_grid = grid;
  t_block = block;
  t_shared = shared;
  t_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = t_grid;
  *block = t_block;
  *shared = t_shared;
  *stream = t_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) { return launch(f); }
hipError_t hipLaunchCooperativeKernel(const void* f, dim3, dim3, void**, unsigned, hipStream_t) {
  return launch(f);
}

hipError_t hipMalloc(void** out, size_t bytes) { return allocate(out, bytes); }
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> hold(state().lock);
  if (p && state().live.erase(static_cast<char*>(p)) == 0) return hipErrorInvalidValue;
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** out, size_t bytes, unsigned) {
  *out = std::calloc(1, bytes > 0 ? bytes : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind) {
  return copy(to, from, bytes);
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind, hipStream_t) {
  return copy(to, from, bytes);
}
hipError_t hipMemsetAsync(void* to, int value, size_t bytes, hipStream_t) {
  if (bytes > 0 && !to) return hipErrorInvalidValue;
  std::memset(to, value, bytes);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
  *free_bytes = *total = size_t{288} << 30;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** out, const void*) {
  static void* p = std::calloc(1, 64 << 20);
  *out = p;
  return hipSuccess;
}

hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* out, hipDeviceAttribute_t what, int) {
  *out = what == hipDeviceAttributeMultiprocessorCount ? 256 : 1024;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* out, int) {
  std::memset(out, 0, sizeof(*out));
  std::strcpy(out->gcnArchName, "gfx950");
  out->warpSize = 64;
  out->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* out, const void*, int, size_t) {
  *out = 2;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* out, unsigned) {
  *out = handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* out) {
  *out = handle<hipEvent_t>();
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* out, unsigned) { return hipEventCreate(out); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* out, hipEvent_t, hipEvent_t) {
  *out = 0.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* out) {
  *out = handle<hipGraph_t>();
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* out, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *out = handle<hipGraphExec_t>();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  std::lock_guard<std::mutex> hold(state().lock);
  state().launched.push_back("graph");
  t_launched.push_back("graph");
  return hipSuccess;
}

}  // extern "C"
