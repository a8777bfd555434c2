// A program whose hipHostMalloc can be made to fail (it stands before the runtime's): frames,
// large reads and ray queries of a context that gets no pinned memory, against those of one
// that does. Prints "ok ..." with the number of refused allocations, "no device" and exits 2
// without a GPU, or the first difference.
#include <dlfcn.h>

#include <cstdio>
#include <cstring>
#include <vector>

#include "trt.h"

static bool g_refuse = false;
static int g_refused = 0;

extern "C" int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  typedef int (*Malloc)(void**, size_t, unsigned);
  static const Malloc real = reinterpret_cast<Malloc>(dlsym(RTLD_NEXT, "hipHostMalloc"));
  if (!g_refuse && real) return real(p, bytes, flags);
  ++g_refused;
  *p = nullptr;
  return 2;  // hipErrorOutOfMemory
}

struct Results {
  std::vector<float> color, hits;
  std::vector<uint8_t> shown, occluded;
  std::vector<uint32_t> inst;
  trt_stats stats;
};

#define OK(call)                                                                                   \
  do {                                                                                             \
    const trt_status s_ = (call);                                                                  \
    if (s_ != TRT_OK) {                                                                            \
      std::printf("FAIL %s: %d %s\n", #call, int(s_), ctx ? trt_last_error(ctx) : "");             \
      return false;                                                                                \
    }                                                                                              \
  } while (0)

static bool use(const char* scene, Results& r) {
  trt_context* ctx = nullptr;
  OK(trt_create(0, &ctx));
  trt_build_opts bo{32, 4, 0, 1.0f};
  trt_scene_file_info info;
  OK(trt_load_scene_file(ctx, scene, &bo, &info));
  trt_render_opts o{};
  o.width = 700;  // 7.8 MB as floats: a threaded read
  o.height = 701;
  o.spp = 2;
  o.max_depth = 4;
  o.rr_depth = 3;
  o.seed = 3;
  o.ray_epsilon = 1e-3f;
  OK(trt_render(ctx, &o, &r.stats));
  r.color.resize(size_t(o.width) * o.height * 4);
  OK(trt_read_color(ctx, r.color.data()));
  trt_tonemap_opts tm{};
  tm.exposure = 1.f;
  tm.gamma = 2.2f;
  r.shown.resize(size_t(o.width) * o.height * 4);
  OK(trt_tonemap(ctx, &tm, r.shown.data()));
  for (const uint32_t n : {1u, 700u, 4096u, 4097u, 20000u}) {
    std::vector<float> rays(size_t(n) * 8);
    uint32_t seed = n;
    for (size_t i = 0; i < rays.size(); ++i) {
      seed = seed * 1664525u + 1013904223u;
      rays[i] = float(seed >> 8) * 0x1p-23f - 1.f;
      if (i % 8 == 3) rays[i] = 0.f;
      if (i % 8 == 7) rays[i] = 1e30f;
    }
    const size_t at = r.inst.size();
    r.hits.resize((at + n) * 4);
    r.inst.resize(at + n);
    r.occluded.resize(at + n);
    OK(trt_trace_closest(ctx, rays.data(), n, &r.hits[at * 4], &r.inst[at]));
    OK(trt_trace_any(ctx, rays.data(), n, &r.occluded[at]));
    rays[3] = -1.f;
    if (trt_trace_any(ctx, rays.data(), n, &r.occluded[at]) != TRT_INVALID_ARG) return std::printf("FAIL invalid ray\n"), false;
  }
  OK(trt_render(ctx, &o, &r.stats));  // and once more with what was allocated on the way
  trt_destroy(ctx);
  return true;
}

int main(int argc, char** argv) {
  if (argc < 2) return 1;
  trt_context* probe = nullptr;
  if (trt_create(0, &probe) != TRT_OK) return std::printf("no device\n"), 2;
  trt_destroy(probe);
  Results with, without;
  if (!use(argv[1], with)) return 1;
  g_refuse = true;
  if (!use(argv[1], without)) return 1;
  if (g_refused == 0) return std::printf("FAIL no allocation was refused\n"), 1;
  const trt_stats &a = with.stats, &b = without.stats;
  if (a.paths != b.paths || a.primary_rays != b.primary_rays || a.extend_rays != b.extend_rays || a.shadow_rays != b.shadow_rays)
    return std::printf("FAIL ray counts\n"), 1;
  if (with.color != without.color || with.shown != without.shown) return std::printf("FAIL images\n"), 1;
  if (std::memcmp(with.hits.data(), without.hits.data(), with.hits.size() * 4) || with.inst != without.inst ||
      with.occluded != without.occluded)
    return std::printf("FAIL ray queries\n"), 1;
  std::printf("ok %d %llu\n", g_refused, static_cast<unsigned long long>(a.extend_rays));
  return 0;
}
