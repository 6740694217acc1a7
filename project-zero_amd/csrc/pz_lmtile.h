// pz_lmtile.h -- which LM-head path and tile shape a call takes (host only).
#pragma once
#include <stddef.h>

// Weights the Infinity Cache (256 MB) cannot hold from one call to the next
// are loaded non-temporally: 128256 x 2560 at batch 1 114 -> 98 us, at 8
// (matrix cores) 116 -> 107; 50257 x 1024, which it can hold, 18.2 -> 19.5.
inline bool lm_once(int V, int n) { return (size_t)V * n * 2 > ((size_t)256 << 20); }

// One tile shape of the GEMM: its batch block, rows per workgroup (one
// workgroup per CU, by LDS), and the time of one round of workgroups on every
// CU at n = 2560 (us, measured at V = 128256).
struct LmTile {
  int cols, rows;
  float round_us;
};
constexpr LmTile LM_TILE_SHAPES[] = {
    {256, 256, 192.0f}, {128, 256, 107.0f}, {64, 256, 83.0f}, {32, 256, 64.0f},
    {16, 256, 59.0f}};
constexpr int LM_TILE_COUNT = sizeof(LM_TILE_SHAPES) / sizeof(LM_TILE_SHAPES[0]);

// The shape with the least time for nb batch rows: rounds of workgroups times
// a round's time.  most: batch rows the workspace holds (a multiple of 16).
inline int lm_tile_for(int V, int nb, int most, int n_cu) {
  int best = LM_TILE_COUNT - 1;
  float best_us = __builtin_inff();
  for (int i = 0; i < LM_TILE_COUNT; i++) {
    const LmTile& t = LM_TILE_SHAPES[i];
    if ((nb + t.cols - 1) / t.cols * t.cols > most) continue;  // parts past the workspace
    const long wgs = (long)((V + t.rows - 1) / t.rows) * ((nb + t.cols - 1) / t.cols);
    const float us = (float)((wgs + n_cu - 1) / n_cu) * t.round_us;
    if (us < best_us) {
      best = i;
      best_us = us;
    }
  }
  return best;
}

// Batches of 4 to 32 whose workgroups make the parts themselves: where the
// launch that makes them once takes longer than it saves.  One round of
// 256-row workgroups: rows of up to 256 (us, own / once, as the kernel that
// staged the parts in every workgroup before: 4 x 128 x 8000 5.4 / 7.9, 5.6;
// 32 x 256 x 50257 12.5 / 13.4, 13.7; but 32 x 512 x 50257 18.3 / 17.2, 21.5).
// More rounds, where a ring per workgroup also fills and drains too often: up
// to 1024, past the Infinity Cache 768 (32 x 256 x 128256 15.6 / 20.7, 20.9;
// fused 32 x 1024 x 128256 44.0 / 48.3, 46.1; 16 x 768 x 200000 68.7 / 74.9,
// 75.0; but 32 x 1024 x 200000 107.7 / 99.3, 109.6).
inline bool lm_own_parts(int V, int n, int B, int n_cu) {
  if (B > 32) return false;
  if (V <= 256 * n_cu) return n <= 256;
  return n <= (lm_once(V, n) ? 768 : 1024);
}
