// net_plan: reads "images H W" lines, writes the rows of a chunk, the blocks per
// image and their bound.
#include <cstdio>

#include "sbp_corr_plan.hpp"

int main()
{
  int nb, H, W;
  while (std::scanf("%d %d %d", &nb, &H, &W) == 3)
    std::printf("%d %ld %ld\n", net_chunk_rows(nb, H, W), net_blocks_per_image(nb, H, W), net_most_blocks(H, W));
  return 0;
}
