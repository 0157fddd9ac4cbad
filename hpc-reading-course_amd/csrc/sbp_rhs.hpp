// sbp_rhs.hpp -- one right-hand side of a small 2D problem from and to vectors
// in host memory, in one launch: a block reads the points its patch and stencils
// need (sbp_step.hpp) straight from the caller-order vector in pinned memory,
// evaluates the patch in LDS and writes its values back, rows of consecutive
// doubles both ways.  Latency bounds it: 65^2 acoustics, order 4, 27 us per
// call against 30 with the two conversions as launches of their own (33^2 21 /
// 25, 101^2 39 / 40; most of either is the processor copying in and out).
#pragma once
#include "sbp_step.hpp"

namespace sbp {

constexpr int kRhsWaves = 4, kRhsRows = 16;  // waves of a block, most rows it loads

// LDS values pass between lanes of one wave: what any lane wrote before is read
// as written by any lane after.  A wave's LDS operations complete in order, so
// the fences cost no wait; they keep the compiler, to which the barrier alone
// says nothing about memory, from moving the accesses across it.
__device__ __forceinline__ void wave_handover()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int ORDER, int PHYS, int MAT>
__global__ __launch_bounds__(64 * kRhsWaves) void rhs_patch_kernel(StepArgs<T> a, double c5, const double *__restrict__ in,
                                                                   double *__restrict__ out)
{
  using Pt = Patch<T, ORDER, PHYS, MAT, false, kRhsWaves, kRhsRows, 1>;
  constexpr int C = Pt::C, KR = Pt::KR;
  __shared__ T s_[step_lds(ORDER, C, kRhsRows)];
  __shared__ double so[kRhsWaves][C * kStepLanes];
  const int i0 = (blockIdx.x % a.px) * a.pw, j0 = (blockIdx.x / a.px) * a.ph;
  const int i1 = min(i0 + a.pw, a.nx);
  const Pt pt(a, s_, i0, i1, j0, min(j0 + a.ph, a.ny));

  // lanes take consecutive values of a row, so that it crosses the link in
  // whole lines; every load is issued before the first is used
  const int n = (pt.xh[0] - pt.xl[0]) * C;
  double v[KR][C];
#pragma unroll
  for (int k = 0; k < KR; k++) {
    const double *row = in + ((long)pt.row(k) * a.nx + pt.xl[0]) * C;
#pragma unroll
    for (int c = 0; c < C; c++) v[k][c] = row[min(pt.lane + kStepLanes * c, n - 1)];
  }
  T ri[KR], Kb[KR];
#pragma unroll
  for (int k = 0; k < KR; k++) {
    ri[k] = Kb[k] = T(1);
    if constexpr (MAT == M_ARR) {
      const long o = pt.at(pt.row(k));
      ri[k] = (Pt::AC ? a.rinv : a.velx)[o];
      Kb[k] = (Pt::AC ? a.bulk : a.vely)[o];
    }
  }
#pragma unroll
  for (int k = 0; k < KR; k++)
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int q = pt.lane + kStepLanes * c, col = q / C, f = q - col * C;
      if (q < n) pt.s[f * Pt::FS + (pt.wv + kRhsWaves * k) * kStepLanes + col] = T(v[k][c]);
    }
  __syncthreads();

  auto rows = [&](auto XE) {
#pragma unroll
    for (int k = 0; k < KR; k++) {
      const int r = pt.wv + kRhsWaves * k, j = pt.yl[0] + r;
      if (j < pt.yl[1] || j >= pt.yh[1]) continue;  // (the whole wave)
      T Yc[C], F[C];
#pragma unroll
      for (int c = 0; c < C; c++) Yc[c] = pt.slot(0, r)[c * Pt::FS];
      pt.template rhs<decltype(XE)::value>(0, r, j, Yc, ri[k], Kb[k], c5, F);
      // a row of results that only this wave writes and reads
      double *o = so[pt.wv];
      if (pt.own()) {
        const int col = pt.xl[0] + pt.lane - i0;
#pragma unroll
        for (int c = 0; c < C; c++) o[col * C + c] = F[c];
      }
      wave_handover();
      double *row = out + ((long)j * a.nx + i0) * C;
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int q = pt.lane + kStepLanes * c;
        if (q < (i1 - i0) * C) row[q] = o[q];
      }
      wave_handover();
    }
  };
  if (pt.xedge) rows(std::true_type{});
  else rows(std::false_type{});
}

// Patches as high as a block loads, at most 10 rows: low ones would read their
// neighbours' rows again over the link.
template <int ORDER> inline StepPlan rhs_plan_t(int nx, int ny)
{
  StepPlan best{};
  for (int ph = 10; ph >= 1 && !best.ok; ph--) best = patch_plan<ORDER>(nx, ny, 1, kRhsRows, ph, ph);
  return best;
}
inline StepPlan rhs_plan(int order, int nx, int ny)
{
  return order == 2 ? rhs_plan_t<2>(nx, ny) : (order == 4 ? rhs_plan_t<4>(nx, ny) : rhs_plan_t<6>(nx, ny));
}

template <typename T, int ORDER, int PHYS, int MAT>
hipError_t rhs_launch(const void *args, double c5, const double *in, double *out, int grid, hipStream_t s)
{
  hipLaunchKernelGGL((rhs_patch_kernel<T, ORDER, PHYS, MAT>), dim3(grid), dim3(64 * kRhsWaves), 0, s,
                     *static_cast<const StepArgs<T> *>(args), c5, in, out);
  return hipGetLastError();
}

template <typename T, int ORDER> RhsLaunchFn pick_rhs(int phys, int mat)
{
  if (phys == PH_ACOUSTIC && mat == M_UNIT) return &rhs_launch<T, ORDER, PH_ACOUSTIC, M_UNIT>;
  if (phys == PH_ACOUSTIC && mat == M_ARR) return &rhs_launch<T, ORDER, PH_ACOUSTIC, M_ARR>;
  if (phys == PH_ACOUSTIC && mat == M_REF) return &rhs_launch<T, ORDER, PH_ACOUSTIC, M_REF>;
  if (phys == PH_ADV2D && mat == M_UNIT) return &rhs_launch<T, ORDER, PH_ADV2D, M_UNIT>;
  if (phys == PH_ADV2D && mat == M_ARR) return &rhs_launch<T, ORDER, PH_ADV2D, M_ARR>;
  return nullptr;
}

}  // namespace sbp
