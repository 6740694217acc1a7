// pz_take_slots (pz_slots.h) on allocators with a given room: the counts it
// ends on, one line each.
#include <cstdio>

#include "pz_slots.h"

static int run(int want, size_t each, size_t free_bytes, size_t room, int* tries) {
  *tries = 0;
  return pz_take_slots(
      want, 32, free_bytes, [=](int n) { return each * (size_t)n; },
      [=](int n) { return ++*tries, each * (size_t)n <= room; });
}

int main() {
  const size_t MiB = (size_t)1 << 20, GiB = MiB << 10;
  const struct {
    const char* what;
    int want;
    size_t each, free_bytes, room;
    int got, tries;
  } cases[] = {
      {"plenty", 256, 4 * MiB, 288 * GiB, 288 * GiB, 256, 1},
      {"a batch below one per CU", 70, 4 * MiB, 288 * GiB, 288 * GiB, 70, 1},
      {"a nearly full device", 256, 4 * MiB, 8 * GiB, 8 * GiB, 32, 1},
      {"a nearly full device, want between", 70, 4 * MiB, 8 * GiB, 8 * GiB, 32, 1},
      {"half of it fits a 64th", 256, 4 * MiB, 40 * GiB, 40 * GiB, 128, 1},
      {"one allocation fails", 256, 4 * MiB, 288 * GiB, 600 * MiB, 128, 2},
      {"less than 32 fit", 256, 4 * MiB, 100 * MiB, 100 * MiB, 16, 2},
      {"only one fits", 256, 4 * MiB, 5 * MiB, 5 * MiB, 1, 6},
      {"one wanted", 1, 4 * MiB, 5 * MiB, 5 * MiB, 1, 1},
      {"none fits", 256, 4 * MiB, 1 * MiB, 1 * MiB, 0, 6},
  };
  int bad = 0;
  for (const auto& c : cases) {
    int tries = 0;
    const int got = run(c.want, c.each, c.free_bytes, c.room, &tries);
    const bool ok = got == c.got && tries == c.tries;
    std::printf("%s: %d after %d tries%s\n", c.what, got, tries, ok ? "" : "  WRONG");
    bad += !ok;
  }
  return bad != 0;
}
