// FP32 right-hand sides on vectors in host memory, order-6 SBP operators (built without FMA contraction).
#include "sbp_rhs.hpp"
namespace sbp {
RhsLaunchFn rhs_launcher_o6_f32(int phys, int mat) { return pick_rhs<float, 6>(phys, mat); }
}  // namespace sbp
