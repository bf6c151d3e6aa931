// fake_hip.cpp -- see fake_hip.hpp.
#include "fake_hip.hpp"

#include <hip/hip_runtime.h>
#include <malloc.h>
#include <stdlib.h>
#include <string.h>

#include <deque>
#include <new>

namespace fake {
namespace {
struct Copy {
  void* dst;
  const void* src;
  size_t bytes;
  hipMemcpyKind kind;
};
// (allocations of this file are not counted: `quiet` is set around them)
bool quiet = false;
struct Quiet {
  bool was = quiet;
  Quiet() { quiet = true; }
  ~Quiet() { quiet = was; }
};
struct Range {
  const char* at;
  size_t bytes;
};
std::deque<Copy> queue;
std::vector<Range> pinned;
long left[kKinds] = {0, 0, 0};
bool hit[kKinds] = {false, false, false};

bool fails(Kind k) {
  if (left[k] == 0 || --left[k] != 0) return false;
  hit[k] = true;
  return true;
}
bool is_pinned(const void* p) {
  for (const Range& r : pinned)
    if (p >= r.at && p < r.at + r.bytes) return true;
  return false;
}
const void* host_side(const Copy& c) {
  const void* p = c.kind == hipMemcpyHostToDevice ? c.src : c.kind == hipMemcpyDeviceToHost ? c.dst : nullptr;
  return p && !is_pinned(p) ? p : nullptr;
}
void drain() {
  for (const Copy& c : queue) memcpy(c.dst, c.src, c.bytes);
  queue.clear();
}
}  // namespace

std::vector<Launch> launches;
size_t freed_under_copy = 0;

size_t pending_host_copies() {
  size_t n = 0;
  for (const Copy& c : queue) n += host_side(c) != nullptr;
  return n;
}
void fail_nth(Kind kind, long n) {
  left[kind] = n;
  hit[kind] = false;
}
bool failed(Kind kind) { return hit[kind]; }

static void* take(size_t n) {
  if (!quiet && fails(kNew)) return nullptr;
  return malloc(n ? n : 1);
}
static void give(void* p) {
  if (!p) return;
  const char* at = static_cast<const char*>(p);
  const size_t n = malloc_usable_size(p);
  for (const Copy& c : queue) {
    const char* h = static_cast<const char*>(host_side(c));
    if (h && h < at + n && at < h + c.bytes) {
      freed_under_copy++;
      return;  // (left allocated, so that the queued copy stays defined)
    }
  }
  free(p);
}
}  // namespace fake

void* operator new(size_t n) {
  void* p = fake::take(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void* operator new[](size_t n) { return operator new(n); }
void* operator new(size_t n, const std::nothrow_t&) noexcept { return fake::take(n); }
void* operator new[](size_t n, const std::nothrow_t&) noexcept { return fake::take(n); }
void operator delete(void* p) noexcept { fake::give(p); }
void operator delete[](void* p) noexcept { fake::give(p); }
void operator delete(void* p, size_t) noexcept { fake::give(p); }
void operator delete[](void* p, size_t) noexcept { fake::give(p); }
void operator delete(void* p, const std::nothrow_t&) noexcept { fake::give(p); }
void operator delete[](void* p, const std::nothrow_t&) noexcept { fake::give(p); }

using fake::Quiet;

extern "C" {
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 160 * 1024;
  return hipSuccess;
}
hipError_t hipDeviceGetName(char* name, int n, hipDevice_t) {
  strncpy(name, "fake", n);
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "made to fail"; }

hipError_t hipMalloc(void** p, size_t n) {
  *p = aligned_alloc(256, (n + 255) & ~(size_t)255);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  Quiet q;
  hipMalloc(p, n);
  fake::pinned.push_back({static_cast<char*>(*p), n});
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  for (size_t i = 0; i < fake::pinned.size(); i++)
    if (fake::pinned[i].at == p) fake::pinned.erase(fake::pinned.begin() + i);
  free(p);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
  Quiet q;
  if (fake::fails(fake::kCopy)) return hipErrorUnknown;
  fake::queue.push_back({dst, src, n, kind});
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  Quiet q;
  fake::drain();
  return hipSuccess;
}

hipError_t hipModuleLoad(hipModule_t* m, const char*) {
  *m = reinterpret_cast<hipModule_t>(8);
  return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
  *f = reinterpret_cast<hipFunction_t>(strdup(name));  // kept: a function lives as long as its module
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by,
                                 unsigned bz, unsigned lds, hipStream_t, void**, void**) {
  Quiet q;
  if (fake::fails(fake::kLaunch)) return hipErrorLaunchFailure;
  fake::launches.push_back({reinterpret_cast<const char*>(f), {gx, gy, gz}, bx * by * bz, lds});
  return hipSuccess;
}
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) {
  *n = 2;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(8);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(8);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  Quiet q;
  if (fake::fails(fake::kLaunch)) return hipErrorLaunchFailure;
  fake::launches.push_back({"graph", {1, 1, 1}, 1, 0});
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
}
