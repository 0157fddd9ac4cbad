// sbp_ctx.hpp -- the single-problem context shared by the host translation
// units (C-ABI, learned corrector).
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/sbp_hip.h"
#include "sbp_kernels.hpp"
#include "sbp_step.hpp"
#include "sbp_xfer.hpp"

struct sbp_ctx {
  sbp_problem d{};
  int C = 0, order = 0, cls = 0, phys = 0, mat = 0, bc = 0, prec = 0;
  int nx = 0, ny = 0, pitch = 0, xoff = 0;
  long plane = 0;
  size_t esz = 8;
  double hix = 0, hiy = 0;
  void *U = nullptr, *A = nullptr, *Y0 = nullptr, *Y1 = nullptr, *KC = nullptr, *TK = nullptr;
  // (TK: 1D Kahan, the compensation of the state in Y0)
  void *rinv = nullptr, *bulk = nullptr;
  void *velx = nullptr, *vely = nullptr;  // advection velocity fields (per-point a, b)
  double *xs = nullptr, *ys = nullptr, *c3x = nullptr, *s3x = nullptr, *c4y = nullptr, *s4y = nullptr;
  // AoS FP64 staging: pinned host memory (aos_host) or device memory (sbp_xfer.hpp); aos2: second operand, on first use
  double *aos = nullptr, *aos2 = nullptr;
  bool aos_host = false;
  sbp::host::Staging staging;
  double *partials = nullptr, *scalar = nullptr;
  int npartials = 0;
  hipStream_t stream = nullptr;
  sbp::StageLaunchFn launch = nullptr;
  sbp::LineLaunchFn line_launch = nullptr;  // 1D: whole steps
  sbp::LaunchGeom geom{};
  int ty_rows = 32, tiles_x = 0, tiles_y = 0, n_tiles = 0, n_edge = 0, n_edge_blocks = 0;
  bool have_state = false;
  // Two-stage interior path (2D acoustics, unit or array materials): pair
  // launcher, D = CLS + R deep frame, tile geometry of the pair tiles.
  sbp::PairLaunchFn pair_launch = nullptr;
  bool fused = false;
  // Whole steps in one launch (sbp_step.hpp), in place of either schedule
  // unless one was chosen with sbp_set_fused (until sbp_reset_schedule).
  sbp::StepLaunchFn step_launch = nullptr;
  sbp::StepPlan step_plan{}, rkf_plan{};
  // one right-hand side of vectors in host memory in one launch (sbp_rhs.hpp)
  sbp::RhsLaunchFn rhs_launch = nullptr;
  sbp::StepPlan rhs_plan{};
  double *rhs_out = nullptr;  // its result (behind aos in its allocation)
  bool whole = false;
  // whole steps march along the grid (sbp_march.hpp)
  sbp::MarchFns march_fns{};
  sbp::MarchPlan march_plan{};
  bool march = false;
  int store_policy = 0;  // two-stage tile stores: 0 by streamed size, 1 cached, 2 nontemporal
  int p_depth = 0, p_ty_rows = 0, p_tiles_x = 0, p_n_tiles = 0, p_n_edge = 0, p_n_edge_blocks = 0;
  // Captured multi-step graphs, keyed by dt and by the array holding U when
  // the capture started (the two-stage path swaps U and Y2 every step).
  struct GraphSlot {
    hipGraphExec_t exec = nullptr;
    double dt = 0;
    void *u = nullptr;
  };
  GraphSlot gslot[2];
  int g_next = 0;
  hipEvent_t ev[5] = {};
  int device = 0;
  void *rkw[8] = {};  // adaptive RK workspace (K1..K6, stage input, candidate), allocated on first use
  double *rk_host = nullptr;  // sums of squared scaled errors of an attempt (pinned host memory)
};


namespace sbp {
namespace host {
// Launch one RK4 stage / one whole step of a context (sbp_capi.hip).
hipError_t launch_step(sbp_ctx *c, double t, double dt);
// H-weighted energy of a planar state laid out like the context's registers
// (U and optional compensation); result left in c->scalar (device) and, when
// out != nullptr, copied to the host.
int energy_of(sbp_ctx *c, const void *u, const void *comp, double *out);
// dst = F(t, src) on planar registers of the context (the RHS stage kernels).
hipError_t launch_rhs(sbp_ctx *c, double t, const void *src, void *dst);
// What steps on chip take of an FP64 context.
StepArgs<double> step_args(const sbp_ctx *c);
// Forget the captured step graph (after the state register moved).
void drop_step_graph(sbp_ctx *c);
}  // namespace host
}  // namespace sbp
