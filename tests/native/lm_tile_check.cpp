// The LM head's path for calls of V ids, n weights and B batch rows, one per
// argument triple: per call a line of "own" (the workgroups make the parts
// themselves) or, per GEMM launch, the tile's index with "nt" where W is read
// non-temporally; first the number of tiles.
#include <cstdio>
#include <cstdlib>

#include "pz_lmtile.h"

int main(int argc, char** argv) {
  const int n_cu = 256, rows = 256;  // compute units; batch rows of one launch
  std::printf("%d\n", LM_TILE_COUNT);
  for (int a = 1; a + 2 < argc; a += 3) {
    const int B = std::atoi(argv[a]), V = std::atoi(argv[a + 1]), n = std::atoi(argv[a + 2]);
    const size_t fit = (size_t)rows * 8192 * 3 / ((size_t)((n + 63) / 64) * 64 * 3) / 16 * 16;
    if (fit == 0 || lm_own_parts(V, n, B, n_cu)) {
      std::printf("own%d\n", B <= 16 ? 16 : 32);
      continue;
    }
    const int most = fit < (size_t)rows ? (int)fit : rows;
    for (int b0 = 0; b0 < B; b0 += most) {
      const int i = lm_tile_for(V, B - b0 < most ? B - b0 : most, most, n_cu);
      std::printf("%d%s ", i, lm_once(V, n) && LM_TILE_SHAPES[i].cols <= 128 ? "nt" : "");
    }
    std::printf("\n");
  }
}
