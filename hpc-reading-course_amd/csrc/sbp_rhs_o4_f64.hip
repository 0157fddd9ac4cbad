// FP64 right-hand sides on vectors in host memory, order-4 SBP operators (built without FMA contraction).
#include "sbp_rhs.hpp"
namespace sbp {
RhsLaunchFn rhs_launcher_o4_f64(int phys, int mat) { return pick_rhs<double, 4>(phys, mat); }
}  // namespace sbp
