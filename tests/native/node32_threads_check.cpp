// Check of trt::pack_nodes32 where threads run out: this program's pthread_create fails from a
// given call on. Every such packing equals that of a single thread. Prints "ok", or the first
// violation and exits non-zero (an escaping exception aborts it).
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "bvh_build.h"

using namespace trt;

static std::atomic<int> g_left{1 << 30};  // threads that may still be created

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  typedef int (*Create)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create real = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
  return g_left.fetch_sub(1) > 0 ? real(t, a, f, arg) : EAGAIN;
}

int main() {
  const uint32_t n = 120000;
  std::mt19937 rng(2);
  std::uniform_real_distribution<float> u(0.f, 1.f);
  std::vector<float> box(size_t(n) * 6);
  for (uint32_t i = 0; i < n; ++i)
    for (int k = 0; k < 3; ++k) {
      box[size_t(i) * 6 + k] = u(rng);
      box[size_t(i) * 6 + 3 + k] = box[size_t(i) * 6 + k] + 0.01f * u(rng);
    }
  const std::vector<DevNode2> dn = to_device_layout(build_binned_sah(box.data(), n, 32, 1, 1, kTravCostTriangles));
  if (dn.size() < 5 * 16384) return std::printf("FAIL %zu nodes are too few for threads\n", dn.size()), 1;
  NodeSpace g{};
  std::vector<DevNode32> one(dn.size());
  if (!pack_nodes32(dn, 0, dn.size(), g, one.data(), 1)) return std::printf("FAIL tree refused\n"), 1;
  for (int threads = 0; threads < 5; ++threads) {
    NodeSpace h{};
    std::vector<DevNode32> some(dn.size());
    g_left = threads;
    const bool ok = pack_nodes32(dn, 0, dn.size(), h, some.data(), 8);
    if (!ok || std::memcmp(&g, &h, sizeof(g)) || std::memcmp(one.data(), some.data(), one.size() * sizeof(DevNode32)))
      return std::printf("FAIL %d threads to be had: another packing\n", threads), 1;
  }
  std::printf("ok\n");
  return 0;
}
