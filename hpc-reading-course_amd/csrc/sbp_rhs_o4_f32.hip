// FP32 right-hand sides on vectors in host memory, order-4 SBP operators (built without FMA contraction).
#include "sbp_rhs.hpp"
namespace sbp {
RhsLaunchFn rhs_launcher_o4_f32(int phys, int mat) { return pick_rhs<float, 4>(phys, mat); }
}  // namespace sbp
