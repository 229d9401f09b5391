// A HIP runtime on the CPU for host code that moves data through streams and
// events: several devices, streams that run nothing before they are waited
// for (so a missing wait shows as wrong data), events that belong to the
// device they were made on (recording one on another device's stream is an
// error, as HIP documents).  Kernels run as loops over their threads.
#pragma once
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#define __host__
#define __device__
#define __global__
#define __launch_bounds__(...)

enum hipError_t { hipSuccess = 0, hipErrorInvalidHandle = 400 };
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipHostMallocPortable = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct double2 { double x, y; };
struct int2 { int x, y; };
inline double2 make_double2(double x, double y) { return {x, y}; }

namespace fake {
inline int device = 0;
struct Stream {
  int device;
  std::vector<std::function<void()>> work;
  size_t done = 0;
  void run(size_t upto) {
    for (; done < upto; done++) work[done]();
  }
};
struct Event {
  int device;
  Stream* stream = nullptr;
  size_t at = 0;
};
inline thread_local dim3 block, thread;
}  // namespace fake
#define blockIdx (fake::block)
#define threadIdx (fake::thread)

typedef fake::Stream* hipStream_t;
typedef fake::Event* hipEvent_t;
typedef void* hipGraph_t;
typedef void* hipGraphExec_t;

inline const char* hipGetErrorString(hipError_t e) { return e ? "invalid handle" : "no error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
template <typename T>
hipError_t hipMalloc(T** p, size_t n) {
  *p = (T*)malloc(n);
  return hipSuccess;
}
template <typename T>
hipError_t hipHostMalloc(T** p, size_t n, unsigned) {
  *p = (T*)aligned_alloc(64, n);
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new fake::Event{fake::device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  e->stream = s;
  e->at = s->work.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->stream) e->stream->run(e->at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  s->run(s->work.size());
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* h, size_t n, hipMemcpyKind, hipStream_t s) {
  std::vector<char> copy((const char*)h, (const char*)h + n);  // pageable: read at once
  s->work.push_back([=]() { memcpy(d, copy.data(), n); });
  return hipSuccess;
}
template <typename K, typename... A>
void hipLaunchKernelGGL(K k, dim3 g, dim3 b, size_t, hipStream_t s, A... a) {
  s->work.push_back([=]() {
    for (fake::block.x = 0; fake::block.x < g.x; fake::block.x++)
      for (fake::thread.x = 0; fake::thread.x < b.x; fake::thread.x++) k(a...);
  });
}
