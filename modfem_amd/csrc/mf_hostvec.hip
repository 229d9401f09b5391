// Host vectors of the C API: between a caller's memory, in the reference's
// row order, and device vectors in the problem's own order.
//
// What bounds it: PCIe.  A copy from pageable memory runs at 35 GB/s towards
// the device and 18 GB/s back, a permutation on one host core at 7 GB/s, a
// core's copy into pinned memory at 75 GB/s and a kernel that reads or writes
// pinned memory at the link's 54 GB/s.  So a vector goes through 1 MB slots
// of a pinned ring: the host fills a slot while a kernel moves the last one,
// and that kernel carries out the permutation on its device side.  912,673
// doubles there and back around a product: 3.9 ms with the permutation on the
// host, pageable copies and allocations, 0.6 ms so.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>

#include "mf_device.h"

namespace mf {

namespace {

// the ring is one per process: 4 MB, whatever the number of problems.  A
// slot is written again only when the kernel that used it last has ended.  It
// belongs to the library stream: when mf_init has chosen another device since
// the last vector, the former stream is waited for and the events, which
// belong to that stream's device, are made anew
constexpr long long kChunk = 1 << 17;  // doubles per slot
constexpr int kSlots = 4;

struct Ring {
  std::mutex m;
  double* p = nullptr;
  hipEvent_t ev[kSlots] = {};
  enum State { kFree, kQueued, kTimed } st[kSlots] = {};  // kTimed: ev tells when it is done
  int next = 0;
  hipStream_t owner = nullptr;

  int init() {
    if (p && owner == stream()) return 0;
    if (owner && owner != stream()) {
      MF_HIP(hipStreamSynchronize(owner));
      all_free();
      owner = nullptr;
      for (hipEvent_t& e : ev) {
        if (e) MF_HIP(hipEventDestroy(e));
        e = nullptr;
      }
    }
    for (hipEvent_t& e : ev)
      if (!e) MF_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (!p) MF_HIP(hipHostMalloc(&p, kSlots * kChunk * sizeof(double), hipHostMallocPortable));
    owner = stream();
    return 0;
  }
  void all_free() {
    for (State& s : st) s = kFree;
  }
  int wait(int s) {
    if (st[s] == kQueued) {
      MF_HIP(hipStreamSynchronize(stream()));
      all_free();
    } else if (st[s] == kTimed) {
      MF_HIP(hipEventSynchronize(ev[s]));
      st[s] = kFree;
    }
    return 0;
  }
  int queued(int s, bool timed) {
    st[s] = kQueued;
    MF_HIP(hipGetLastError());
    if (timed) {
      MF_HIP(hipEventRecord(ev[s], stream()));
      st[s] = kTimed;
    }
    return 0;
  }
};

Ring g_ring;

}  // namespace

// two entries per thread; h and (without iperm) d are 16-byte aligned
__global__ void __launch_bounds__(256) k_vec_in(int n, const double* h, const int* iperm,
                                                double* d) {
  const int i = 2 * (blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  if (i + 1 < n) {
    const double2 v = *reinterpret_cast<const double2*>(h + i);
    if (iperm) {
      const int2 p = *reinterpret_cast<const int2*>(iperm + i);
      d[p.x] = v.x;
      d[p.y] = v.y;
    } else {
      *reinterpret_cast<double2*>(d + i) = v;
    }
  } else {
    d[iperm ? iperm[i] : i] = h[i];
  }
}

__global__ void __launch_bounds__(256) k_vec_out(int n, const double* d, const int* iperm,
                                                 double* h) {
  const int i = 2 * (blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  if (i + 1 < n) {
    double2 v;
    if (iperm) {
      const int2 p = *reinterpret_cast<const int2*>(iperm + i);
      v = make_double2(d[p.x], d[p.y]);
    } else {
      v = *reinterpret_cast<const double2*>(d + i);
    }
    *reinterpret_cast<double2*>(h + i) = v;
  } else {
    h[i] = d[iperm ? iperm[i] : i];
  }
}

static dim3 vec_grid(int n) { return dim3((n + 511) / 512); }

int vec_to_device(const double* h, const int* d_iperm, int n, double* d) {
  std::lock_guard<std::mutex> lock(g_ring.m);
  if (g_ring.init()) return -2;
  for (long long o = 0; o < n; o += kChunk) {
    const int cnt = (int)std::min<long long>(kChunk, n - o), s = g_ring.next;
    if (g_ring.wait(s)) return -2;
    double* slot = g_ring.p + s * kChunk;
    std::memcpy(slot, h + o, (size_t)cnt * sizeof(double));
    hipLaunchKernelGGL(k_vec_in, vec_grid(cnt), dim3(256), 0, stream(), cnt, slot,
                       d_iperm ? d_iperm + o : nullptr, d_iperm ? d : d + o);
    if (g_ring.queued(s, n > kChunk)) return -2;
    g_ring.next = (s + 1) % kSlots;
  }
  return 0;
}

int vec_to_host(const double* d, const int* d_iperm, int n, double* h) {
  std::lock_guard<std::mutex> lock(g_ring.m);
  if (g_ring.init()) return -2;
  const int nch = (int)((n + kChunk - 1) / kChunk);
  const int first = g_ring.next;
  auto count = [&](int c) { return (int)std::min<long long>(kChunk, n - c * kChunk); };
  auto issue = [&](int c) -> int {
    const int s = (first + c) % kSlots;
    if (g_ring.wait(s)) return -2;
    const long long o = c * kChunk;
    hipLaunchKernelGGL(k_vec_out, vec_grid(count(c)), dim3(256), 0, stream(), count(c),
                       d_iperm ? d : d + o, d_iperm ? d_iperm + o : nullptr,
                       g_ring.p + s * kChunk);
    return g_ring.queued(s, nch > 1);
  };
  for (int c = 0; c < std::min(nch, kSlots); c++)
    if (issue(c)) return -2;
  for (int c = 0; c < nch; c++) {
    const int s = (first + c) % kSlots;
    if (g_ring.wait(s)) return -2;
    std::memcpy(h + c * kChunk, g_ring.p + s * kChunk, (size_t)count(c) * sizeof(double));
    if (c + kSlots < nch && issue(c + kSlots)) return -2;
  }
  g_ring.next = (first + nch) % kSlots;
  g_ring.all_free();  // one stream: what was queued before the last slot is done too
  return 0;
}

// the problem's row order on the device: made for the first host vector
int host_order(Problem& P) {
  std::lock_guard<std::mutex> lock(P.vecs.m);
  if (P.d_iperm) return 0;
  int* p = nullptr;
  MF_HIP(hipMalloc(&p, (size_t)P.n * sizeof(int)));
  if (hipMemcpyAsync(p, P.setup.iperm.data(), (size_t)P.n * sizeof(int), hipMemcpyHostToDevice,
                     stream()) != hipSuccess ||
      hipStreamSynchronize(stream()) != hipSuccess) {
    (void)hipFree(p);
    set_error("host vectors: copy of the row order failed");
    return -2;
  }
  P.d_iperm = p;
  return 0;
}

int VecPool::take(int n, double** d) {
  {
    std::lock_guard<std::mutex> lock(m);
    if (!kept.empty()) {
      *d = kept.back();
      kept.pop_back();
      return 0;
    }
  }
  MF_HIP(hipMalloc(d, std::max<size_t>(n, 1) * sizeof(double)));
  return 0;
}

void VecPool::give(double* d) {
  {
    std::lock_guard<std::mutex> lock(m);
    if (kept.size() < kKeep) {
      kept.push_back(d);
      return;
    }
  }
  (void)hipFree(d);
}

void VecPool::release() {
  std::lock_guard<std::mutex> lock(m);
  for (double* d : kept) (void)hipFree(d);
  kept.clear();
}

}  // namespace mf
