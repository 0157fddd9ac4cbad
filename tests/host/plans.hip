// plans: reads "order nx ny resident" lines, writes march_plan's strips, segments,
// rows of a segment, and the frame's patches.  Compiled for the host alone.
#include <cstdio>

#include "sbp_step.hpp"

int main()
{
  int order, nx, ny, resident;
  while (std::scanf("%d %d %d %d", &order, &nx, &ny, &resident) == 4) {
    const int px = sbp::step_plan(order, nx, ny).px;
    const sbp::MarchPlan p = sbp::march_plan(order, nx, ny, px, resident);
    std::printf("%d %d %d %d %d\n", p.ok, p.strips, p.segs, p.seg_rows, sbp::march_frame(order, px, ny));
  }
  return 0;
}
