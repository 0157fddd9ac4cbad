// FP64 marched whole steps of the order-4 SBP operators (built without FMA contraction).
#include "sbp_march.hpp"
namespace sbp {
MarchFns march_launcher_o4_f64(int phys, int mat) { return pick_march<double, 4, false>(phys, mat); }
BatchLaunchFn batch_march_launcher_o4_f64(int mat) { return pick_batch_march<double, 4, false>(mat); }
}  // namespace sbp
