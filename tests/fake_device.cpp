// A device made of host memory, for CPU tests of the host layer: the entry points
// of the kernel library that a device manager calls, each done when it is called.
// Loaded with global visibility before the host library, whose references bind here.
// The three kernels of an image stem keep what the tests look at, the bytes they
// read: the layout pass hands its image through, the convolution copies its input.
#include "glow_mi355x.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

struct mi355x_graph {
  std::vector<std::function<void()>> nodes;
};
struct mi355x_arena {
  std::vector<uint8_t> bytes[3];
};

namespace {
thread_local mi355x_graph *g_capture = nullptr;
// (a recorded launch keeps its arguments, as the real one does)
int launch(std::function<void()> f) {
  if (g_capture) g_capture->nodes.push_back(std::move(f));
  else f();
  return MI355X_OK;
}
int8_t quantized(float x, float scale, int32_t offset) {
  const float r = std::nearbyint(x / scale + (float)offset);
  return r != r ? 0 : (int8_t)std::max(-128.0f, std::min(127.0f, r));
}
int handle(void **p) {
  *p = std::malloc(sizeof(long));
  return MI355X_OK;
}
std::atomic<long> g_replays{0};
// FAKE_DEVICE_MEET: a launch waits until as many threads are inside one
bool met() {
  static std::atomic<int> inside{0};
  const char *n = std::getenv("FAKE_DEVICE_MEET");
  inside++;
  for (int i = 0; n && inside < std::atoi(n); i++) {
    if (i == 20000) return false;
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
  }
  return true;
}
} // namespace

extern "C" {

const char *mi355x_last_error(void) { return "fake device"; }
int mi355x_num_devices(int *n) { *n = 1; return MI355X_OK; }
int mi355x_init(int) { return MI355X_OK; }
int mi355x_set_device(int, int *previous) { if (previous) *previous = 0; return MI355X_OK; }
int mi355x_device_info(mi355x_info *info) {
  std::memset(info, 0, sizeof *info);
  info->total_memory = info->free_memory = 1ull << 32;
  return MI355X_OK;
}
int mi355x_malloc(void **p, size_t n) { *p = std::malloc(n); return MI355X_OK; }
int mi355x_free(void *p) { std::free(p); return MI355X_OK; }
int mi355x_host_alloc(void **p, size_t n) {
  const char *most = std::getenv("FAKE_DEVICE_PINNED_MOST");   // bytes of one allocation
  if (most && n > std::strtoull(most, nullptr, 10)) return MI355X_ERR_RUNTIME;
  *p = std::aligned_alloc(4096, (n + 4095) & ~(size_t)4095);
  return MI355X_OK;
}
int mi355x_host_free(void *p) { std::free(p); return MI355X_OK; }
int mi355x_host_is_pinned(const void *, int *pinned) { *pinned = 0; return MI355X_OK; }
int mi355x_memcpy_h2d(void *d, const void *s, size_t n, void *) { std::memcpy(d, s, n); return MI355X_OK; }
int mi355x_memcpy_d2h(void *d, const void *s, size_t n, void *) { std::memcpy(d, s, n); return MI355X_OK; }
int mi355x_fill_u8(void *d, int v, size_t n, void *) { return launch([=] { std::memset(d, v, n); }); }
int mi355x_copy_u8(void *d, const void *s, size_t n, void *) { return launch([=] { std::memcpy(d, s, n); }); }

int mi355x_copy_segments(const mi355x_copy_segment *s, size_t n, uint32_t *done, uint32_t value,
                         uint32_t *, void *) {
  for (size_t i = 0; i < n; i++) {
    if (s[i].op != MI355X_SEGMENT_COPY) return MI355X_ERR_NOT_SUPPORTED;
    std::memcpy(s[i].dst, s[i].src, s[i].bytes);
  }
  if (done) *done = value;
  return MI355X_OK;
}

int mi355x_stream_create(void **p) { return handle(p); }
int mi355x_stream_destroy(void *p) { std::free(p); return MI355X_OK; }
int mi355x_stream_sync(void *) { return MI355X_OK; }
int mi355x_stream_query(void *, int *idle) { *idle = 1; return MI355X_OK; }
int mi355x_stream_wait_event(void *, void *) { return MI355X_OK; }
int mi355x_event_create(void **p) { return handle(p); }
int mi355x_event_destroy(void *p) { std::free(p); return MI355X_OK; }
int mi355x_event_record(void *e, void *) { *(long *)e = g_replays; return MI355X_OK; }
int mi355x_event_sync(void *) { return MI355X_OK; }
// A graph takes a millisecond, launches one by one FAKE_DEVICE_DIRECT_MS.
int mi355x_event_elapsed_ms(void *a, void *b, float *ms) {
  const char *direct = std::getenv("FAKE_DEVICE_DIRECT_MS");
  *ms = direct && *(long *)a == *(long *)b ? (float)std::atof(direct) : 1.0f;
  return MI355X_OK;
}
long fake_graph_launches(void) { return g_replays; }

int mi355x_graph_begin_capture(void *) { g_capture = new mi355x_graph; return MI355X_OK; }
int mi355x_graph_end_capture(void *, mi355x_graph **g) { *g = g_capture; g_capture = nullptr; return MI355X_OK; }
int mi355x_graph_launch(mi355x_graph *g, void *) { g_replays++; for (auto &f : g->nodes) f(); return MI355X_OK; }
int mi355x_graph_destroy(mi355x_graph *g) { delete g; return MI355X_OK; }

int mi355x_arena_create(size_t c, size_t m, size_t a, mi355x_arena **out) {
  *out = new mi355x_arena;
  const size_t sizes[3] = {c, m, a};
  for (int i = 0; i < 3; i++) (*out)->bytes[i].assign(sizes[i] + 256, 0xA5);
  return MI355X_OK;
}
int mi355x_arena_destroy(mi355x_arena *a) { delete a; return MI355X_OK; }
int mi355x_arena_ptr(mi355x_arena *a, int region, size_t offset, void **p) {
  *p = a->bytes[region].data() + offset;
  return MI355X_OK;
}
int mi355x_arena_upload(mi355x_arena *a, int region, size_t offset, const void *s, size_t n, void *) {
  std::memcpy(a->bytes[region].data() + offset, s, n);
  return MI355X_OK;
}
uint64_t mi355x_arena_bytes(const mi355x_arena *a) {
  return a->bytes[0].size() + a->bytes[1].size() + a->bytes[2].size();
}

int mi355x_quantize_i8(int8_t *d, const float *s, size_t n, float scale, int32_t offset, void *) {
  return launch([=] { for (size_t i = 0; i < n; i++) d[i] = quantized(s[i], scale, offset); });
}
int mi355x_rowsum_i8(int32_t *, const int8_t *, size_t, size_t, void *) { return MI355X_OK; }
int mi355x_space_to_depth2_i8(int8_t *d, const int8_t *s, size_t N, size_t IH, size_t IW, size_t C,
                              size_t, size_t, size_t BH, size_t BW, size_t Cout, int32_t, void *) {
  return launch([=] { std::memcpy(d, s, std::min(N * IH * IW * C, N * BH * BW * Cout)); });
}
int mi355x_quantize_space_to_depth2_i8(int8_t *d, const float *s, size_t N, size_t IH, size_t IW,
                                       size_t C, size_t, size_t, size_t BH, size_t BW, size_t Cout,
                                       int32_t, float scale, int32_t offset, void *) {
  return launch([=] {
    for (size_t i = 0; i < std::min(N * IH * IW * C, N * BH * BW * Cout); i++)
      d[i] = quantized(s[i], scale, offset);
  });
}
int mi355x_cwq_conv2d_i8_opts(int8_t *out, const int8_t *in, const int8_t *, const void *, int,
                              const mi355x_conv_geom *geom, int32_t, int32_t, const int32_t *,
                              const int32_t *, const int32_t *, const int32_t *, const int32_t *,
                              const int32_t *, const int32_t *, const int32_t *, int32_t,
                              const int32_t *, int, const int32_t *, void *,
                              const mi355x_launch_opts *) {
  const mi355x_conv_geom g = *geom;
  if (!met()) return MI355X_ERR_RUNTIME;
  return launch([=] {
    std::memcpy(out, in, std::min((size_t)g.N * g.IH * g.IW * g.IC, (size_t)g.N * g.OH * g.OW * g.OC));
  });
}

} // extern "C"
