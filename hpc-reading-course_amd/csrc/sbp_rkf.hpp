// sbp_rkf.hpp -- a whole Runge-Kutta-Fehlberg 4(5) attempt of a 2D problem in
// one launch, in LDS: the six stages of a patch as sbp_step.hpp computes the
// four of RK4.  K1 .. K5 of a lane's points stay in registers, the stage
// operand passes through LDS.  A block leaves its sum of squared scaled errors
// in host memory, where the caller adds them up.  The arithmetic per point is
// that of the separate launches (sbp_rk45_f64.hip), term for term.
//
// What bounds it: a block's chain of six stages with a barrier each, and the
// points evaluated for their neighbours (order 4: 64 x 32 loaded for 40 x 8).
// 201^2, order 4: 27 us per attempt (the kernel 16, then the host's sum and
// decision), thirteen launches 70 (and 90 when the
// error came back through a copy call).
#pragma once
#include "sbp_step.hpp"

namespace sbp {

// Fehlberg's coefficients (E. Fehlberg, NASA TR R-315, 1969).
constexpr double kRkfC[6] = {0.0, 1.0 / 4.0, 3.0 / 8.0, 12.0 / 13.0, 1.0, 1.0 / 2.0};
constexpr double kRkfA[6][5] = {{0, 0, 0, 0, 0},
                                {1.0 / 4.0, 0, 0, 0, 0},
                                {3.0 / 32.0, 9.0 / 32.0, 0, 0, 0},
                                {1932.0 / 2197.0, -7200.0 / 2197.0, 7296.0 / 2197.0, 0, 0},
                                {439.0 / 216.0, -8.0, 3680.0 / 513.0, -845.0 / 4104.0, 0},
                                {-8.0 / 27.0, 2.0, -3544.0 / 2565.0, 1859.0 / 4104.0, -11.0 / 40.0}};
constexpr double kRkfB5[6] = {16.0 / 135.0, 0.0, 6656.0 / 12825.0, 28561.0 / 56430.0, -9.0 / 50.0, 2.0 / 55.0};
constexpr double kRkfB4[6] = {25.0 / 216.0, 0.0, 1408.0 / 2565.0, 2197.0 / 4104.0, -1.0 / 5.0, 0.0};

// rows a block loads: kStepWaves * rkf_rows(order)
constexpr int rkf_rows(int order) { return order == 6 ? 5 : 4; }

struct RkfArgs {
  StepArgs<double> g;  // u: U, uo: the candidate
  double c5[6];        // cos(5 pi t) at the stages' times (M_REF)
  double h, atol, rtol;
  double *partial;  // a value per block
};

template <int ORDER, int PHYS, int MAT>
__global__ __launch_bounds__(64 * kStepWaves) void rkf_patch_kernel(RkfArgs ra)
{
  constexpr int NW = kStepWaves, KR = rkf_rows(ORDER), H = NW * KR;
  using Pt = Patch<double, ORDER, PHYS, MAT, false, NW, H, 6>;
  constexpr int C = Pt::C;
  constexpr bool AC = Pt::AC;
  __shared__ double s_[step_lds(ORDER, C, H)];
  __shared__ double sh[NW];
  const StepArgs<double> &a = ra.g;
  const int i0 = (blockIdx.x % a.px) * a.pw, j0 = (blockIdx.x / a.px) * a.ph;
  const Pt pt(a, s_, i0, min(i0 + a.pw, a.nx), j0, min(j0 + a.ph, a.ny));

  double U[KR][C], K[5][KR][C], ri[KR], Kb[KR];
#pragma unroll
  for (int k = 0; k < KR; k++) {
    const long o = pt.at(pt.row(k));
#pragma unroll
    for (int c = 0; c < C; c++) U[k][c] = a.u[c * a.plane + o];
    ri[k] = Kb[k] = 1.0;
    if constexpr (MAT == M_ARR) {
      ri[k] = (AC ? a.rinv : a.velx)[o];
      Kb[k] = (AC ? a.bulk : a.vely)[o];
    }
  }
#pragma unroll
  for (int k = 0; k < KR; k++)
#pragma unroll
    for (int c = 0; c < C; c++) pt.slot(0, pt.wv + NW * k)[c * Pt::FS] = U[k][c];
  __syncthreads();

  double acc = 0;
  auto stages = [&](auto XE) {
#pragma unroll
    for (int st = 0; st < 6; st++) {
      const int b = st & 1;
#pragma unroll
      for (int k = 0; k < KR; k++) {
        const int r = pt.wv + NW * k, j = pt.yl[0] + r;
        if (j < pt.yl[st + 1] || j >= pt.yh[st + 1]) continue;  // (the whole wave)
        double Yc[C], F[C];
#pragma unroll
        for (int c = 0; c < C; c++) Yc[c] = pt.slot(b, r)[c * Pt::FS];
        pt.template rhs<decltype(XE)::value>(b, r, j, Yc, ri[k], Kb[k], ra.c5[st], F);
        if (st < 5) {
#pragma unroll
          for (int c = 0; c < C; c++) {
            K[st][k][c] = F[c];
            double sum = kRkfA[st + 1][0] * K[0][k][c];
#pragma unroll
            for (int q = 1; q <= st; q++) sum = sum + kRkfA[st + 1][q] * K[q][k][c];
            pt.slot(b ^ 1, r)[c * Pt::FS] = U[k][c] + ra.h * sum;
          }
        } else if (pt.own()) {
          const long o = pt.at(j);
#pragma unroll
          for (int c = 0; c < C; c++) {
            double sb = kRkfB5[0] * K[0][k][c], se = (kRkfB5[0] - kRkfB4[0]) * K[0][k][c];
#pragma unroll
            for (int q = 1; q < 6; q++) {
              const double f = q < 5 ? K[q < 5 ? q : 0][k][c] : F[c];
              sb = sb + kRkfB5[q] * f;
              se = se + (kRkfB5[q] - kRkfB4[q]) * f;
            }
            const double u5 = U[k][c] + ra.h * sb, err = ra.h * se, y4 = u5 - err;
            const double w = err / (ra.atol + ra.rtol * fmax(fabs(u5), fabs(y4)));
            acc += w * w;
            a.uo[c * a.plane + o] = u5;
          }
        }
      }
      __syncthreads();
    }
  };
  if (pt.xedge) stages(std::true_type{});
  else stages(std::false_type{});
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if (pt.lane == 0) sh[pt.wv] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = sh[0];
    for (int w = 1; w < NW; w++) sum += sh[w];
    ra.partial[blockIdx.x] = sum;
  }
}

// an attempt's patches
template <int ORDER> inline StepPlan rkf_plan_t(int nx, int ny)
{
  return patch_plan<ORDER>(nx, ny, 6, kStepWaves * rkf_rows(ORDER), 1, 20);
}
inline StepPlan rkf_plan(int order, int nx, int ny)
{
  return order == 2 ? rkf_plan_t<2>(nx, ny) : (order == 4 ? rkf_plan_t<4>(nx, ny) : rkf_plan_t<6>(nx, ny));
}

template <int ORDER, int PHYS, int MAT> hipError_t rkf_launch(const RkfArgs &a, int grid, hipStream_t s)
{
  hipLaunchKernelGGL((rkf_patch_kernel<ORDER, PHYS, MAT>), dim3(grid), dim3(64 * kStepWaves), 0, s, a);
  return hipGetLastError();
}
using RkfLaunchFn = hipError_t (*)(const RkfArgs &a, int grid, hipStream_t s);
template <int ORDER> RkfLaunchFn pick_rkf(int phys, int mat)
{
  if (phys == PH_ACOUSTIC && mat == M_UNIT) return &rkf_launch<ORDER, PH_ACOUSTIC, M_UNIT>;
  if (phys == PH_ACOUSTIC && mat == M_ARR) return &rkf_launch<ORDER, PH_ACOUSTIC, M_ARR>;
  if (phys == PH_ACOUSTIC && mat == M_REF) return &rkf_launch<ORDER, PH_ACOUSTIC, M_REF>;
  if (phys == PH_ADV2D && mat == M_UNIT) return &rkf_launch<ORDER, PH_ADV2D, M_UNIT>;
  if (phys == PH_ADV2D && mat == M_ARR) return &rkf_launch<ORDER, PH_ADV2D, M_ARR>;
  return nullptr;
}
// sbp_rkf_o{2,4,6}_f64.hip
RkfLaunchFn rkf_launcher_o2(int phys, int mat);
RkfLaunchFn rkf_launcher_o4(int phys, int mat);
RkfLaunchFn rkf_launcher_o6(int phys, int mat);

}  // namespace sbp
