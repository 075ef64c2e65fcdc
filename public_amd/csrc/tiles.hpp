// How many grid lines a work-group of a sweep takes (host only).
#pragma once

#include "line_ops.hpp"

namespace cruna {

// The most lines, a power of two up to tl_max, that fill at most wg_max threads
// and divide the lines lying side by side (np: grid of the device layout, d:
// direction of the sweep).
inline int auto_tl(const int *np, int d, int wg_max, int tl_max) {
  const long lines_contig = d == 0 ? (long)np[1] * np[2] : np[0];
  const int NB = np[d] / PPT;
  int TL = 1;
  while (NB * TL * 2 <= wg_max && lines_contig % (TL * 2) == 0 && TL * 2 <= tl_max) TL *= 2;
  return TL;
}

constexpr long GPU_CUS = 256;

// Lines per work-group of the sweeps along d where the caller names none;
// wg_max: the kernels' largest work-group.
// x-lines are contiguous: up to 256 threads; y/z tiles take up to 16
// neighbouring x-lines (128-byte rows in FP64) in up to wg_max threads.
// FP64 grids with less than a wavefront per SIMD (1024): work-groups of one
// wavefront where its lines fill it, spread over more CUs (a step with filters,
// x alone: 32^3 169 -> 155 us, 60 x 65 x 70 481 -> 471; 64^3 228 -> 224, y and z
// alone 225 each).  Along y and z a wavefront of long lines has few of them, and
// with less than 8 (64-byte rows) each row's cache lines are fetched by several
// work-groups: such tiles are widened, up to 16 lines, while a work-group per
// CU remains.  Steps in us with a wavefront / 4 / 8 / 16 lines (* taken):
//   64 x 32 x 128 (4)  231 /    - / 228* / 238      64 x 64 x 128 (4)  327 /   - / 315 / 311*
//   32 x 32 x 256 (2)  253 / 238* / 244 / 269       64 x 32 x 256 (2)  368 / 323 / 313* / 336
//   16 x 16 x 256 (2)  183* / 187 / 197 / 225       16 x 64 x 512 (1)  472 / 329* / 344 / -
inline int auto_tile_lines(const int *np, int d, bool fp64, int wg_max) {
  const long N = (long)np[0] * np[1] * np[2];
  const int NB = np[d] / PPT;
  const bool small = fp64 && N <= 1024L * 64 * PPT && 64 % NB == 0;
  if (d == 0) return auto_tl(np, d, small ? 64 : 256, 1 << 20);
  const int most = auto_tl(np, d, wg_max, 16);
  if (!small) return most;
  int TL = auto_tl(np, d, 64, 16);
  if (TL < 8)
    while (TL * 2 <= most && N / (np[d] * TL * 2L) >= GPU_CUS) TL *= 2;
  return TL;
}

}  // namespace cruna
