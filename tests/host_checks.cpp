// Checks of the host layer's C++ interface that its C view does not reach (no GPU
// needed); each prints what it found and returns 0, or 1 when it does not hold.
#include "../glow_amd/host/Backend.h"
#include "../glow_amd/host/Staging.h"

#include <cfenv>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <sched.h>

using namespace glow_mi355x;

static int bag_offsets() {
  const int32_t lengths[] = {3, -5, 0, 7, INT32_MAX, 4};
  const std::vector<int32_t> want = {0, 3, 3, 3, 10, INT32_MAX, INT32_MAX, INT32_MAX};
  return MI355XFunction::bagOffsets(lengths, 6, 7) == want ? 0 : 1;
}

// Values on the rounding ties and below the smallest normal number, quantized under the
// caller's rounding mode and with denormals flushed: by the caller alone, and together
// with the helper threads of a pool made under that mode.
static int quantized_under(int mode, unsigned flush) {
  const size_t n = 4 * kStagePiece / sizeof(float) + 77;   // with what no vector takes
  std::vector<float> x(n);
  std::vector<int8_t> want(n);
  for (int part = 0; part < 2; part++) {
    const float scale = part ? 1e-41f : 0.5f;
    for (size_t i = 0; i < n; i++) {
      x[i] = (float)((int)(i % 401) - 200) * scale * 0.5f;
      want[i] = (int8_t)std::max(-128.0f, std::min(127.0f, std::nearbyint(x[i] / scale + 3.0f)));
    }
    for (size_t bytes : {n * sizeof(float), (size_t)4 * 333}) {
      const unsigned before = __builtin_ia32_stmxcsr();
      std::fesetround(mode);
      __builtin_ia32_ldmxcsr(__builtin_ia32_stmxcsr() | flush);
      StagingPool pool;
      const std::unique_ptr<uint8_t, decltype(&std::free)> staged(
          (uint8_t *)std::aligned_alloc(4096, (n + 4095) / 4096 * 4096), &std::free);   // as pinned memory is
      std::vector<StagePiece> pieces;
      for (size_t at = 0; at < bytes; at += kStagePiece) {
        StagePiece p;
        p.src = (const uint8_t *)x.data() + at;
        p.bytes = std::min(kStagePiece, bytes - at);
        p.form = StagePiece::Quantized;
        p.scale = scale;
        p.offset = 3.0f;
        p.at = at / 4;
        pieces.push_back(p);
      }
      pool.run(pieces, staged.get(), [](size_t, size_t) { return (int)MI355X_OK; });
      const bool kept = std::fegetround() == mode && (__builtin_ia32_stmxcsr() & 0x8040) == flush;
      __builtin_ia32_ldmxcsr(before);
      std::fesetround(FE_TONEAREST);
      if (!kept) return std::printf("the caller's mode has changed\n"), 1;
      for (size_t i = 0; i < bytes / 4; i++)
        if ((int8_t)staged.get()[i] != want[i])
          return std::printf("%zu of %zu: %d, not %d\n", i, bytes / 4, (int8_t)staged.get()[i], want[i]), 1;
    }
  }
  return 0;
}

// A third of three CPUs, whatever the machine has.
static int helpers_of_three_cpus() {
  cpu_set_t all, three;
  CPU_ZERO(&three);
  if (sched_getaffinity(0, sizeof all, &all) != 0) return 2;
  for (int i = 0, n = 0; i < CPU_SETSIZE && n < 3; i++)
    if (CPU_ISSET(i, &all)) CPU_SET(i, &three), n++;
  if (sched_setaffinity(0, sizeof three, &three) != 0) return 2;
  const int n = StagingPool().helpers();
  std::printf("%d helpers\n", n);
  return n <= 1 ? 0 : 1;
}

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "bag_offsets")) return bag_offsets();
  if (!std::strcmp(name, "downward")) return quantized_under(FE_DOWNWARD, 0);
  if (!std::strcmp(name, "upward")) return quantized_under(FE_UPWARD, 0);
  if (!std::strcmp(name, "flushed")) return quantized_under(FE_TONEAREST, 0x8040);
  if (!std::strcmp(name, "helpers_of_three_cpus")) return helpers_of_three_cpus();
  std::printf("no check called %s\n", name);
  return 2;
}
