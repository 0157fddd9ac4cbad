// FP32 and FP32+Kahan marched whole steps of the order-2 SBP operators.
#include "sbp_march.hpp"
namespace sbp {
MarchFns march_launcher_o2_f32(int phys, int mat, bool kahan)
{
  return kahan ? pick_march<float, 2, true>(phys, mat) : pick_march<float, 2, false>(phys, mat);
}
BatchLaunchFn batch_march_launcher_o2_f32(int mat, bool kahan)
{
  return kahan ? pick_batch_march<float, 2, true>(mat) : pick_batch_march<float, 2, false>(mat);
}
}  // namespace sbp
