// The HIP runtime functions that libsfx.so calls, on host memory, for tests of its host code without
// a GPU (test_host_calls.py loads this library before libsfx.so). Kernels do nothing; copies and
// fills are made at once. What is kept is the order of things: per stream (null: the null stream)
// how many operations were issued and how many the host has waited for; allocations, one of which
// can be made to fail; and what k_give_scalars, the kernel that hands the step scalars over, saw.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct Stream { long issued = 0, waited = 0; std::string last; };
struct Event { hipStream_t s = nullptr; long at = 0; };
std::mutex mu;
std::map<hipStream_t, Stream> streams;
std::map<const void*, std::string> kernels;
std::map<void*, size_t> device, pinned;
std::map<std::string, long> launches;
long fail_in = 0, stale = 0, clock_ms = 0, operations = 0;
bool ones = false, capturing = false;
thread_local hipError_t last = hipSuccess;   // until it is asked for, as the real one
std::map<size_t, std::pair<void*, std::vector<char>>> copied;   // by size: the last copy to the device

struct Call { dim3 grid, block; size_t lds; hipStream_t stream; };
thread_local std::vector<Call> calls;

void issue(hipStream_t s, const std::string& what) {
  if (capturing) return;
  ++operations;
  ++streams[s].issued;
  streams[s].last = what;
}
hipError_t take(void** p, size_t n, std::map<void*, size_t>& in) {
  std::lock_guard<std::mutex> lk(mu);
  if (fail_in > 0 && --fail_in == 0) return last = hipErrorOutOfMemory;
  if (!(*p = std::calloc(n, 1))) return hipErrorOutOfMemory;
  in[*p] = n;
  return hipSuccess;
}
hipError_t give(void* p, std::map<void*, size_t>& in) {
  std::lock_guard<std::mutex> lk(mu);
  in.erase(p);
  std::free(p);
  return hipSuccess;
}
void copy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  std::memcpy(d, s, n);
  if (k != hipMemcpyHostToDevice) return;
  auto it = device.find(d);
  if (it == device.end() || it->second != n)   // not a whole allocation: a member of a batch's list
    copied[n] = {d, std::vector<char>((const char*)s, (const char*)s + n)};
}
}  // namespace

extern "C" {
// -------------------------------------------------------------------------- for the tests
// Streams with work that the host has not waited for, their last operations in `what`.
int fake_busy(char* what, int n) {
  std::lock_guard<std::mutex> lk(mu);
  std::string t;
  int k = 0;
  for (auto& s : streams)
    if (s.second.issued > s.second.waited) { ++k; t += (s.first ? "stream: " : "null stream: ") + s.second.last + "; "; }
  std::strncpy(what, t.c_str(), (size_t)n - 1);
  what[n - 1] = 0;
  return k;
}
void fake_settle() { std::lock_guard<std::mutex> lk(mu); for (auto& s : streams) s.second.waited = s.second.issued; }
long fake_live(int pins) { std::lock_guard<std::mutex> lk(mu); return (long)(pins ? pinned : device).size(); }
long fake_bytes() {
  std::lock_guard<std::mutex> lk(mu);
  long n = 0;
  for (auto& d : device) n += (long)d.second;
  return n;
}
void fake_fail(long in) { std::lock_guard<std::mutex> lk(mu); fail_in = in; }
// The scalars handed over from now on: every word 1 (an unstable step), or what was there.
void fake_ones(int on) { std::lock_guard<std::mutex> lk(mu); ones = on != 0; }
// Launches of k_give_scalars that found another descriptor than the last one given to a batch.
long fake_stale() { std::lock_guard<std::mutex> lk(mu); return stale; }
// Launches, copies and fills so far.
long fake_operations() { std::lock_guard<std::mutex> lk(mu); return operations; }
long fake_launches(const char* part) {
  std::lock_guard<std::mutex> lk(mu);
  long n = 0;
  for (auto& k : launches) if (k.first.find(part) != std::string::npos) n += k.second;
  return n;
}

// ------------------------------------------------------------------------------ the runtime
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char room[1 << 16]; *p = room; return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return take(p, n, device); }
hipError_t hipFree(void* p) { return give(p, device); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n, pinned); }
hipError_t hipHostFree(void* p) { return give(p, pinned); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  std::lock_guard<std::mutex> lk(mu);
  ++operations;
  copy(d, s, n, k);
  streams[nullptr].waited = streams[nullptr].issued;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  std::lock_guard<std::mutex> lk(mu);
  copy(d, s, n, k);
  issue(st, "copy");
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {   // need not be finished on return
  std::lock_guard<std::mutex> lk(mu);
  std::memset(p, v, n);
  issue(nullptr, "fill");
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t st) {
  std::lock_guard<std::mutex> lk(mu);
  std::memset(p, v, n);
  issue(st, "fill");
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  streams.erase(s);
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  streams[s].waited = streams[s].issued;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { fake_settle(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Event; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  *(Event*)e = {s, streams[s].issued};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> lk(mu);
  Stream& s = streams[((Event*)e)->s];
  if (s.waited < ((Event*)e)->at) s.waited = ((Event*)e)->at;
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {   // each span is longer than the last
  std::lock_guard<std::mutex> lk(mu);
  *ms = (float)++clock_ms;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capturing = true; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { capturing = false; *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { *x = (hipGraphExec_t)1; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  issue(s, "graph");
  return hipSuccess;
}

void** __hipRegisterFatBinary(const void*) { static void* m; return &m; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  std::lock_guard<std::mutex> lk(mu);
  kernels[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  calls.push_back({g, b, lds, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  const Call c = calls.back();
  calls.pop_back();
  *g = c.grid; *b = c.block; *lds = c.lds; *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  const std::string& k = kernels[f];
  ++launches[k];
  issue(s, k);
  if (k.find("k_give_scalars") == std::string::npos) return hipSuccess;
  void* inst = *(void**)args[0];
  char* out = *(char**)args[4];
  const size_t n = pinned.count(out) ? pinned[out] / grid.x : 0;
  if (ones)
    for (size_t i = 0; i < n / 4; ++i) ((int*)out)[i] = 1;
  auto it = copied.find(device.count(inst) ? device[inst] : 0);
  if (it != copied.end() && it->second.first != inst && std::memcmp(inst, it->second.second.data(), it->first)) ++stale;
  return hipSuccess;
}
}
