// sbp_corr_plan.hpp -- how the corrector's fused kernels cut images into windows
// of columns and chunks of rows (host code; the kernels are in sbp_corr.hip).
#pragma once
#include <algorithm>

constexpr int FW = 64, FOUT = FW - 6;  // window width, output columns
constexpr int FUSED_HALO = 9;          // row steps beyond the chunk's rows
constexpr int FUSED_MAX_ROWS = 32;     // output rows per block (LDS staging)

// Rows of each block's chunk (at most FUSED_MAX_ROWS, chunks as even as
// possible) for nb images.  A block runs its rows and FUSED_HALO more in whole
// groups of six steps; a step takes 0.55 us where a CU has one block and 0.43 us
// per block where it has more.  The split of the least total is taken: tall
// chunks for many images, low ones that spread a few over the chip (64 corrected
// steps of one 257^2 image 4.2 ms with chunks of 29 rows, 3.1 with 9; a training
// step of one 172 and 142 us).  Chunks of n rows are even if some number of them
// makes them so; there are FUSED_MAX_ROWS heights to look at, whatever H.
inline int net_chunk_rows(int nb, int H, int W)
{
  constexpr int kCus = 256;
  const long strips = (long)nb * ((W + FOUT - 1) / FOUT);
  int best = 1;
  double least = 1e300;
  for (int rows = std::min(FUSED_MAX_ROWS, H); rows >= 1; rows--) {
    const int chunks = (H + rows - 1) / rows;
    if ((H + chunks - 1) / chunks != rows) continue;
    const long blocks = strips * chunks;
    const double cost = (rows + FUSED_HALO + 5) / 6 * 6 * std::max(0.55, 0.43 * (double)((blocks + kCus - 1) / kCus));
    if (cost < least) {
      least = cost;
      best = rows;
    }
  }
  return best;
}
inline long net_blocks_per_image(int nb, int H, int W)
{
  const int rows = net_chunk_rows(nb, H, W);
  return (long)((W + FOUT - 1) / FOUT) * ((H + rows - 1) / rows);
}
// at most, for any number of images (chunks of one row)
inline long net_most_blocks(int H, int W) { return (long)((W + FOUT - 1) / FOUT) * H; }
