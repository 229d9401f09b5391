// Host vectors through the pinned ring on the CPU runtime of fake_hip: vectors
// of one and of many slots, to and from two devices in turn, with and without
// a row order.  Prints the first difference and returns 1.
#include "../../modfem_amd/csrc/mf_hostvec.hip"

#include <cstdio>
#include <numeric>
#include <random>

namespace mf {
static hipStream_t g_now = nullptr;
static std::string g_err;
hipStream_t stream() { return g_now; }
void set_error(const std::string& s) { g_err = s; }
}  // namespace mf

using namespace mf;

struct Vec {
  std::vector<double> h;
  std::vector<int> perm;
  double* d = nullptr;
  int dev;
};

int main(int argc, char**) {
  const bool switch_devices = argc > 1;
  fake::Stream st[2] = {{0}, {1}};
  std::mt19937 rng(7);
  std::vector<Vec> all;
  auto fail = [](const char* what, int round) {
    printf("round %d: %s %s\n", round, what, g_err.c_str());
    return 1;
  };
  const int sizes[] = {5, 1 << 17, (1 << 17) + 1, 3, 1000003, 77, 4 << 17, 131071, 600001, 9};
  for (int round = 0; round < 40; round++) {
    const int dev = switch_devices ? (round / 3) % 2 : 0;
    fake::device = dev;
    g_now = &st[dev];
    Vec v;
    v.dev = dev;
    const int n = sizes[rng() % 10];
    v.h.resize(n);
    for (double& x : v.h) x = (double)rng();
    if (round % 2) {
      v.perm.resize(n);
      std::iota(v.perm.begin(), v.perm.end(), 0);
      std::shuffle(v.perm.begin(), v.perm.end(), rng);
    }
    if (hipMalloc(&v.d, n * sizeof(double))) return 1;
    std::vector<double> sent = v.h;
    if (vec_to_device(sent.data(), v.perm.empty() ? nullptr : v.perm.data(), n, v.d))
      return fail("to the device:", round);
    std::fill(sent.begin(), sent.end(), -1.0);  // read on return
    all.push_back(std::move(v));
    if (round % 4 == 3) {  // one of this device's vectors back
      for (size_t k = all.size(); k-- > 0;)
        if (all[k].dev == dev) {
          const Vec& w = all[k];
          std::vector<double> got(w.h.size(), -2.0);
          if (vec_to_host(w.d, w.perm.empty() ? nullptr : w.perm.data(), (int)w.h.size(), got.data()))
            return fail("to the host:", round);
          if (got != w.h) return fail("wrong vector", round);
          break;
        }
    }
  }
  // what every device holds once its stream has run
  for (fake::Stream& s : st) s.run(s.work.size());
  for (size_t k = 0; k < all.size(); k++) {
    const Vec& v = all[k];
    for (size_t i = 0; i < v.h.size(); i++)
      if (v.d[v.perm.empty() ? i : v.perm[i]] != v.h[i]) return fail("wrong on the device", (int)k);
  }
  printf("ok\n");
  return 0;
}
