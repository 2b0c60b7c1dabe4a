// Checks of the host layer's C++ interface that its C view does not reach (no GPU
// needed); each prints what it found and returns 0, or 1 when it does not hold.
#include "../glow_amd/host/Backend.h"

#include <cstdio>
#include <cstring>

using namespace glow_mi355x;

static int bag_offsets() {
  const int32_t lengths[] = {3, -5, 0, 7, INT32_MAX, 4};
  const std::vector<int32_t> want = {0, 3, 3, 3, 10, INT32_MAX, INT32_MAX, INT32_MAX};
  return MI355XFunction::bagOffsets(lengths, 6, 7) == want ? 0 : 1;
}

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "bag_offsets")) return bag_offsets();
  std::printf("no check called %s\n", name);
  return 2;
}
