// FP32 right-hand sides on vectors in host memory, order-2 SBP operators (built without FMA contraction).
#include "sbp_rhs.hpp"
namespace sbp {
RhsLaunchFn rhs_launcher_o2_f32(int phys, int mat) { return pick_rhs<float, 2>(phys, mat); }
}  // namespace sbp
