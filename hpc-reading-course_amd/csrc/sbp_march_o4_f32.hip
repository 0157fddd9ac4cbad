// FP32 and FP32+Kahan marched whole steps of the order-4 SBP operators.
#include "sbp_march.hpp"
namespace sbp {
MarchFns march_launcher_o4_f32(int phys, int mat, bool kahan)
{
  return kahan ? pick_march<float, 4, true>(phys, mat) : pick_march<float, 4, false>(phys, mat);
}
BatchLaunchFn batch_march_launcher_o4_f32(int mat, bool kahan)
{
  return kahan ? pick_batch_march<float, 4, true>(mat) : pick_batch_march<float, 4, false>(mat);
}
}  // namespace sbp
