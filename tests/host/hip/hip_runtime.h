// A stand-in for the HIP runtime on the host, for checks of what
// fivonagi_amd/csrc/fv_runtime.cpp asks of it (tests/host/runtime_check.cpp).
// Device memory is host memory (large blocks are address space alone, and copies
// from and to them move nothing); work on streams is done when they are waited
// for, launches and captured launches at once; a call can be made to fail.
#ifndef FAKE_HIP_RUNTIME_H
#define FAKE_HIP_RUNTIME_H

#include <stddef.h>
#include <stdint.h>
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2,
                     hipErrorInvalidHandle = 400,
                     hipErrorStreamCaptureUnsupported = 900;

namespace fake {
struct Stream {
  int device;
  std::vector<std::function<void()>> queued;   // copies not yet done
};
struct Event { int device; };
struct Graph { std::vector<std::function<void()>> nodes; };
constexpr size_t kLarge = 256u << 20;          // from this size on memory is never touched
struct State {
  std::recursive_mutex mu;
  Stream null_stream{0, {}};
  std::vector<Stream*> streams;
  Stream* capturing = nullptr;                 // the stream under capture, by anyone
  Graph* into = nullptr;
  std::map<void*, size_t> blocks;
  bool no_pinned = false;                      // hipHostMalloc fails
  int fail_copy = -1;                          // asynchronous copies until one fails (< 0: none)
  std::vector<float> elapsed;                  // hipEventElapsedTime's answers, in turn
  size_t asked = 0;
};
inline int& device() { static thread_local int d = 0; return d; }
inline State& st() { static State s; return s; }
inline bool real(const void* p) {              // not in a large block
  auto it = st().blocks.upper_bound((void*)p);
  if (it == st().blocks.begin()) return true;
  --it;
  return it->second < kLarge || (const char*)p >= (const char*)it->first + it->second;
}
inline void launch(std::function<void()> f) {
  std::lock_guard<std::recursive_mutex> lk(st().mu);
  if (st().into) st().into->nodes.push_back(f);
  else f();
}
}  // namespace fake

typedef fake::Stream* hipStream_t;
typedef fake::Event* hipEvent_t;
typedef fake::Graph* hipGraph_t;
typedef fake::Graph* hipGraphExec_t;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum { hipDeviceAttributeMultiprocessorCount, hipStreamNonBlocking, hipStreamCaptureModeThreadLocal,
       hipEventDisableTiming, hipHostMallocDefault, hipHostMallocPortable };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive };
#define FAKE_LOCK std::lock_guard<std::recursive_mutex> lk_(fake::st().mu)

inline const char* hipGetErrorString(hipError_t) { return "fake"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = fake::device(); return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::device() = d; return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return hipSuccess; }
inline hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)1 << 38; return hipSuccess; }

inline hipError_t fake_alloc(void** p, size_t n) {
  FAKE_LOCK;
  *p = n >= fake::kLarge ? mmap(nullptr, n, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0)
                         : std::calloc(n ? n : 1, 1);
  fake::st().blocks[*p] = n;
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  FAKE_LOCK;
  auto it = fake::st().blocks.find(p);
  if (it == fake::st().blocks.end()) std::abort();
  if (it->second >= fake::kLarge) munmap(p, it->second);
  else std::free(p);
  fake::st().blocks.erase(it);
  return hipSuccess;
}
template <class T> hipError_t hipMalloc(T** p, size_t n) { return fake_alloc((void**)p, n); }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  return fake::st().no_pinned ? hipErrorOutOfMemory : fake_alloc(p, n);
}
inline hipError_t hipHostFree(void* p) { return hipFree(p); }

inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  FAKE_LOCK;
  if (fake::real(d) && fake::real(s)) std::memmove(d, s, n);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  FAKE_LOCK;
  auto& g = fake::st();
  if (g.fail_copy >= 0 && g.fail_copy-- == 0) return hipErrorInvalidValue;
  if (fake::real(d) && fake::real(s))
    (st ? st : &g.null_stream)->queued.push_back([=] { std::memmove(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  FAKE_LOCK;
  if (fake::real(d)) std::memset(d, v, n);
  return hipSuccess;
}
inline hipError_t hipMemset(void* d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }

inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  FAKE_LOCK;
  *s = new fake::Stream{fake::device(), {}};
  fake::st().streams.push_back(*s);
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
  FAKE_LOCK;
  auto& v = fake::st().streams;
  for (size_t k = 0; k < v.size(); ++k)
    if (v[k] == s) v.erase(v.begin() + k);
  delete s;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  FAKE_LOCK;
  if (!s) s = &fake::st().null_stream;
  if (fake::st().capturing == s) return hipErrorStreamCaptureUnsupported;
  for (auto& f : s->queued) f();
  s->queued.clear();
  return hipSuccess;
}
inline hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* v) {
  *v = s && fake::st().capturing == s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
inline hipError_t hipStreamBeginCapture(hipStream_t s, int) {
  FAKE_LOCK;
  if (fake::st().capturing) return hipErrorStreamCaptureUnsupported;
  fake::st().capturing = s;
  fake::st().into = new fake::Graph;
  return hipSuccess;
}
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  FAKE_LOCK;
  *g = fake::st().into;
  fake::st().capturing = nullptr;
  fake::st().into = nullptr;
  return hipSuccess;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t) {
  *e = new fake::Graph(*g);
  return hipSuccess;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (auto& f : e->nodes) fake::launch(f);
  return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return hipSuccess; }

inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new fake::Event{fake::device()};
  return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (s && e->device != s->device) return hipErrorInvalidHandle;
  return hipStreamSynchronize(s);                // an event's work is done when it is recorded
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  auto& g = fake::st();
  *ms = g.asked < g.elapsed.size() ? g.elapsed[g.asked] : 1e3f;
  ++g.asked;
  return hipSuccess;
}

#endif  // FAKE_HIP_RUNTIME_H
