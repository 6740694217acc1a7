// pz_slots.h -- how many of a set of equal buffers a sampler takes.
#pragma once
#include <stddef.h>

// Tries take(n), which allocates n buffers and says whether it could, from
// n = want down by halves (but not past `modest`), passing over counts above
// `modest` whose bytes(n) exceed a 64th of the free memory; returns the first
// n taken, or 0.
// (One buffer per CU serves most, every count is correct, and a sampler must
// neither fail to be made for want of the large ones nor take what a nearly
// full device has left.)
template <class Bytes, class Take>
int pz_take_slots(int want, int modest, size_t free_bytes, Bytes bytes, Take take) {
  for (int n = want; n > 0; n = n > modest && n / 2 < modest ? modest : n / 2) {
    if (n > modest && bytes(n) > free_bytes / 64) continue;
    if (take(n)) return n;
  }
  return 0;
}
