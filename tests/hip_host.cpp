// The HIP runtime calls of the library's host code, on the CPU, for tests of what that code asks for: device
// memory is host memory, kernels are counted and not run.  Work on a stream waits until something
// synchronises with it, the latest that the runtime may do it, so that memory which is released or reused
// without a wait is seen to be.  Loaded with its symbols global before the library.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>
#include <thread>
#include <vector>

struct ihipEvent_t {
  hipStream_t stream = nullptr;
  uint64_t op = 0;   // the event is the op of this number on that stream
  uint64_t kernel = 0;   // and the kernel of this number
};

struct ihipStream_t {
  struct Op {
    void* dst;
    const void* src;
    size_t n;               // a copy, n > 0
    hipStream_t after;      // or a wait for another stream
    uint64_t after_op, after_kernel;
  };
  std::deque<Op> queue;
  uint64_t kernel = 0, kernel_done = 0;   // the last one launched, and waited for, by their numbers in the process
  uint64_t done = 0;        // ops executed so far
  uint64_t last() const { return done + queue.size(); }
};

namespace {

std::map<const void*, std::string> names;
std::vector<std::string> launched;
std::vector<hipStream_t> streams;
std::map<char*, size_t> allocated;
std::map<char*, uint64_t> allocated_at;   // after this kernel
uint64_t kernels = 0;
int overwritten = 0;
int64_t groups = 0;
size_t most_lds = 0;
int violations = 0, fail_wait_after = -1, wait_us = 0, lds = 160 * 1024;
double elapsed = 0, elapsed_step = 0;
struct Config { dim3 grid, block; size_t shmem; hipStream_t stream; } config;

bool inside(const void* p, const char* base, size_t n) { return (const char*)p >= base && (const char*)p < base + n; }

void run_to(hipStream_t s, uint64_t op) {
  while (s->done < op) {
    const ihipStream_t::Op o = s->queue.front();
    if (o.after) {
      run_to(o.after, o.after_op);
      o.after->kernel_done = std::max(o.after->kernel_done, o.after_kernel);
    }
    if (o.n) memcpy(o.dst, o.src, o.n);
    s->queue.pop_front();
    s->done++;
  }
}

void run_all() {
  for (hipStream_t s : streams) {
    run_to(s, s->last());
    s->kernel_done = s->kernel;
  }
}

// A write to memory that kernels which no one has waited for may read: all but what was allocated after them.
void check_write(const char* p) {
  auto a = allocated.upper_bound((char*)p);
  if (a == allocated.begin() || !(--a, inside(p, a->first, a->second))) return;
  for (hipStream_t s : streams)
    if (s->kernel > s->kernel_done && s->kernel > allocated_at[a->first]) overwritten++;
}

hipError_t allocate(void** p, size_t n) {
  *p = calloc(1, n ? n : 1);
  allocated[(char*)*p] = n;
  allocated_at[(char*)*p] = kernels;
  return hipSuccess;
}

hipError_t release(void* p) {
  const size_t n = allocated[(char*)p];
  int used = 0;
  for (hipStream_t s : streams)
    for (const auto& o : s->queue)
      if (o.n && (inside(o.dst, (char*)p, n) || inside(o.src, (char*)p, n))) used++;
  if (used) run_all();
  violations += used;
  allocated.erase((char*)p);
  free(p);
  return hipSuccess;
}

}  // namespace

extern "C" {

// ---- for the tests
// What the streams still hold; memory released while a copy on it waited.
int hip_host_pending() {
  size_t n = 0;
  for (hipStream_t s : streams) n += s->queue.size();
  return (int)n;
}
int hip_host_violations() { return violations; }
// Memory written from the host while a kernel that may read it waited on a stream.
int hip_host_overwritten() { return overwritten; }
// Streams made so far, and those that have had a transfer.
int hip_host_streams() { return (int)streams.size(); }
int hip_host_used_streams() {
  int n = 0;
  for (hipStream_t s : streams) n += s->last() > 0 ? 1 : 0;
  return n;
}
// The n-th wait for an event from now on fails (-1: none does).
void hip_host_fail_wait(int n) { fail_wait_after = n; }
// Every wait for an event that is not done takes this long.
void hip_host_wait_us(int us) { wait_us = us; }
// The LDS of a workgroup from now on.
void hip_host_lds(int bytes) { lds = bytes; }
// Elapsed times: first, then each smaller than the one before by `step`.
void hip_host_elapsed(double first, double step) { elapsed = first; elapsed_step = step; }
// The kernels launched since the last call, one name a line.
int hip_host_launches(char* out, int len) {
  std::string all;
  for (const std::string& k : launched) all += k + "\n";
  launched.clear();
  snprintf(out, len, "%s", all.c_str());
  return (int)all.size();
}
// The most LDS that a launch has asked for so far.
int64_t hip_host_most_lds() { return (int64_t)most_lds; }
// The workgroups launched since the last call.
int64_t hip_host_groups() {
  const int64_t n = groups;
  groups = 0;
  return n;
}

// ---- the runtime
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : lds;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return allocate(p, n); }
hipError_t hipHostFree(void* p) { return release(p); }
// (the streams do not wait for the null stream, nor it for them)
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { check_write((char*)d); memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { check_write((char*)d); memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = new ihipStream_t;
  streams.push_back(*s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (!s) return hipSuccess;
  run_to(s, s->last());
  s->kernel_done = s->kernel;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { run_all(); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (s && e->stream) s->queue.push_back({nullptr, nullptr, 0, e->stream, e->op, e->kernel});
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* src, size_t n, hipMemcpyKind k, hipStream_t s) {
  if (!s) return hipMemcpy(d, src, n, k);
  s->queue.push_back({d, src, n, nullptr, 0, 0});
  return hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->stream = s;
  e->op = s ? s->last() : 0;
  e->kernel = s ? s->kernel : 0;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (fail_wait_after >= 0 && fail_wait_after-- == 0) return hipErrorUnknown;
  if (!e->stream) return hipSuccess;
  e->stream->kernel_done = std::max(e->stream->kernel_done, e->kernel);
  if (e->stream->done >= e->op) return hipSuccess;
  if (wait_us) std::this_thread::sleep_for(std::chrono::microseconds(wait_us));
  run_to(e->stream, e->op);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = (float)elapsed;
  elapsed *= 1 - elapsed_step;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return hipMalloc(p, (size_t)4 << 20); }

void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  names[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
  config = Config{grid, block, shmem, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
  *grid = config.grid; *block = config.block; *shmem = config.shmem; *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t shmem, hipStream_t s) {
  kernels++;
  if (s) s->kernel = kernels;
  launched.push_back(names[f]);
  most_lds = std::max(most_lds, shmem);
  groups += (int64_t)grid.x * grid.y * grid.z;
  return hipSuccess;
}

}  // extern "C"
