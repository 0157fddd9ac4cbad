// One-launch RKF4(5) attempts of the order-4 SBP operators (built without FMA contraction).
#include "sbp_rkf.hpp"
namespace sbp {
RkfLaunchFn rkf_launcher_o4(int phys, int mat) { return pick_rkf<4>(phys, mat); }
}  // namespace sbp
