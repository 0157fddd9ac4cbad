// One-launch RKF4(5) attempts of the order-6 SBP operators (built without FMA contraction).
#include "sbp_rkf.hpp"
namespace sbp {
RkfLaunchFn rkf_launcher_o6(int phys, int mat) { return pick_rkf<6>(phys, mat); }
}  // namespace sbp
