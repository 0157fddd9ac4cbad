// sbp_step.hpp -- a whole RK4 step of a 2D problem in one launch, in LDS.
//
// A block computes the four stages of one patch of the grid: it loads U on the
// patch grown by what four stages of stencils reach (closure rows read the
// first TAPS points of their line, interior rows R points to either side) and
// evaluates each stage on what the following ones still need.  The region's
// rows are dealt to the waves in turn, one lane per column, so a point's U,
// its running sum (Y2-U) + 2(Y3-U) + (Y4-U) and its materials stay in
// registers, only the stage operand passes through LDS (two buffers, one
// barrier per stage), and whether a row is a closure row is one decision per
// wave.  The arithmetic per point is that of the one-stage kernels, term for
// term, so FP64 results are the same to the bit; U' goes to another array
// (neighbouring patches read U), whose role the host trades with U's.
#pragma once
#include <type_traits>

#include "sbp_kernels.hpp"

namespace sbp {

constexpr int kStepLanes = 64;  // columns of a loaded region, at most
constexpr int kStepWaves = 8;
// rows of a loaded region, at most: kStepWaves * step_rows(order)
constexpr int step_rows(int order) { return order == 6 ? 4 : 3; }

// values of a patch's LDS array: two buffers of every component, and R slots at either end
constexpr int step_lds(int order, int comps, int rows) { return 2 * comps * rows * kStepLanes + order; }

template <typename T> struct StepArgs {
  const T *u;
  T *uo, *comp;  // U'; Kahan compensation (read and written at the patch's own points)
  const T *rinv, *bulk;  // acoustics: rho^-1, K planes (M_ARR)
  const T *velx, *vely;  // 2D advection: velocity planes (M_ARR)
  const double *xs, *ys, *c3x, *s3x, *c4y, *s4y;  // rho = 2 + xy and its forcing (M_REF)
  double c5[3];          // cos(5 pi t) at the times of stage 1, stages 2 and 3, stage 4
  long plane;
  int pitch, xoff, nx, ny, bc;
  T hix, hiy, ax, ay;
  T c12, c3, ca, third;  // dt/2, dt, dt/6, 1/3
  int px, pw, ph;        // patches per row, their width and height
  int strips, segs, seg_rows;  // marched strips (sbp_march.hpp): columns, segments of rows, rows of a segment
};

// The points the stencils of [lo, hi) read along a line of n points.
template <int ORDER> __host__ __device__ inline void stencil_reach(int &lo, int &hi, int n)
{
  using G = Geom<ORDER>;
  const bool l = lo < G::CLS, h = hi > n - G::CLS;
  const int a = l ? 0 : lo - G::R, b = h ? n : hi + G::R;
  lo = h && n - G::TAPS < a ? n - G::TAPS : a;
  hi = l && G::TAPS > b ? G::TAPS : b;
}

// A patch of the grid in a block's LDS array s_: columns [i0, i1) and rows
// [j0, j1), for a method of NST stages, by NW waves, at most H rows loaded.
// TR: "columns" and "rows" are the grid's rows and columns (a narrow strip
// along the left or right boundary fills the lanes that way; it must not reach
// the closure rows at the lanes' ends).
template <typename T, int ORDER, int PHYS, int MAT, bool TR, int NW, int H, int NST> struct Patch {
  using G = Geom<ORDER>;
  static constexpr int R = G::R, CLS = G::CLS, TAPS = G::TAPS, KR = H / NW;
  static constexpr bool AC = PHYS == PH_ACOUSTIC;
  static constexpr int C = AC ? 3 : 1;
  static constexpr int FS = H * kStepLanes, BS = C * FS;  // strides of a field and of a buffer of the LDS array
  static_assert(H % NW == 0 && 2 * BS + 2 * R == step_lds(ORDER, C, H), "rows and LDS of a patch");
  static_assert(!TR || MAT != M_REF, "the forcing's tables are per grid column");

  const StepArgs<T> &a;
  T *const s;  // a lane's x taps may reach R slots outside its row: garbage that no used value depends on
  const int nx, ny;
  const T hl, hr;  // of the lane and row axes
  const int lane, wv;
  // regions evaluated in stages 1 .. NST ([NST]: the patch), and loaded ([0])
  int xl[NST + 1], xh[NST + 1], yl[NST + 1], yh[NST + 1];
  bool xedge, yedge;  // closure columns (rows) among the region's
  int i;
  T cf[TAPS];
  int xt, xpad;
  double xc = 0, c3c = 0, s3c = 0;

  __device__ __forceinline__ Patch(const StepArgs<T> &args, T *s_, int i0, int i1, int j0, int j1)
      : a(args), s(s_ + R), nx(TR ? args.ny : args.nx), ny(TR ? args.nx : args.ny), hl(TR ? args.hiy : args.hix),
        hr(TR ? args.hix : args.hiy), lane(threadIdx.x & 63), wv(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6))
  {
    xl[NST] = i0, xh[NST] = i1, yl[NST] = j0, yh[NST] = j1;
#pragma unroll
    for (int k = NST - 1; k >= 0; k--) {
      xl[k] = xl[k + 1], xh[k] = xh[k + 1], yl[k] = yl[k + 1], yh[k] = yh[k + 1];
      stencil_reach<ORDER>(xl[k], xh[k], nx);
      stencil_reach<ORDER>(yl[k], yh[k], ny);
    }
    xedge = xl[1] < CLS || xh[1] > nx - CLS;
    yedge = yl[1] < CLS || yh[1] > ny - CLS;
    i = min(xl[0] + lane, xh[0] - 1);
    // x taps of this lane: closure columns read a table row from their end of
    // the line; interior ones the interior row, whose padding taps re-read the
    // centre (a point that is certainly valid) with coefficient zero
    xt = lane - R, xpad = lane;
    if (xedge) {
      const bool lo = i < CLS, hi = i >= nx - CLS;
      const int row = lo ? i : (hi ? CLS + (nx - 1 - i) : 2 * CLS);
#pragma unroll
      for (int t = 0; t < TAPS; t++) cf[t] = c_edge<T, ORDER>.c[row][t];
      if (lo || hi) {
        xt = min(max((lo ? 0 : nx - TAPS) - xl[0], 0), kStepLanes - TAPS);
        xpad = -1;
      }
    }
    if constexpr (MAT == M_REF) {
      xc = a.xs[i];
      c3c = a.c3x[i];
      s3c = a.s3x[i];
    }
  }

  // grid row of region row r (clamped: rows past the region repeat its last)
  __device__ __forceinline__ int row(int k) const { return min(yl[0] + wv + NW * k, yh[0] - 1); }
  // offset of this lane's point of row j
  __device__ __forceinline__ long at(int j) const
  {
    return TR ? (long)i * a.pitch + a.xoff + j : (long)j * a.pitch + a.xoff + i;
  }
  __device__ __forceinline__ bool own() const { return xl[0] + lane >= xl[NST] && xl[0] + lane < xh[NST]; }
  __device__ __forceinline__ T *slot(int b, int r) const { return s + b * BS + r * kStepLanes + lane; }

  // Right-hand side at row j = region row r of buffer b, centre values Yc.
  template <bool xe>
  __device__ __forceinline__ void rhs(int b, int r, int j, const T *Yc, T rik, T Kk, double c5, T *K) const
  {
    constexpr int NX = xe ? TAPS : 2 * R + 1;
    const T *f = s + b * BS, *fp = AC ? f + 2 * FS : f;
    // u differentiated in x, v in y, p in both
    const T *fx = f + (TR && AC ? FS : 0) + r * kStepLanes, *px = fp + r * kStepLanes;
    const bool yc = yedge && (j < CLS || j >= ny - CLS);  // closure row
    const int ry = yc ? (j < CLS ? 0 : ny - TAPS) - yl[0] : r - R;
    const T *py = fp + ry * kStepLanes + lane, *vy = f + (TR ? 0 : FS) + ry * kStepLanes + lane;
    // p (or the one field) and u / v along the lanes; p and v / u across
    T ax[NX], bx[NX], ay[TAPS], by[TAPS];
#pragma unroll
    for (int t = 0; t < NX; t++) {
      const int q = xe ? (t < 2 * R + 1 || xpad < 0 ? xt + t : xpad) : lane - R + t;
      ax[t] = px[q];
      if constexpr (AC) bx[t] = fx[q];
    }
#pragma unroll
    for (int t = 0; t < 2 * R + 1; t++) {
      ay[t] = py[t * kStepLanes];
      if constexpr (AC) by[t] = vy[t * kStepLanes];
    }
    if (yc) {
#pragma unroll
      for (int t = 2 * R + 1; t < TAPS; t++) {
        ay[t] = py[t * kStepLanes];
        if constexpr (AC) by[t] = vy[t * kStepLanes];
      }
    }
    const int gi = TR ? j : i, gj = TR ? i : j;  // grid column and row
    auto dlane = [&](const T *v) {
      if constexpr (xe) {
        T acc = cf[0] * v[0];
#pragma unroll
        for (int t = 1; t < TAPS; t++) acc = mad(cf[t], v[t], acc);
        return hl * acc;
      } else {
        return dint<T, ORDER>([&](int t) { return v[t]; }, hl);
      }
    };
    auto drow = [&](const T *v) {
      if (yc) {
        const T *cy = c_edge<T, ORDER>.c[j < CLS ? j : CLS + (ny - 1 - j)];
        T acc = cy[0] * v[0];
#pragma unroll
        for (int t = 1; t < TAPS; t++) acc = mad(cy[t], v[t], acc);
        return hr * acc;
      }
      return dint<T, ORDER>([&](int t) { return v[t]; }, hr);
    };
    if constexpr (AC) {
      const T lp = dlane(ax), rp = drow(ay), lf = dlane(bx), rf = drow(by);
      const T dxp = TR ? rp : lp, dyp = TR ? lp : rp, dxu = TR ? rf : lf, dyv = TR ? lf : rf;
      T fu = T(0), fv = T(0);
      if constexpr (MAT == M_REF) ref_material_at<T>(xc, c3c, s3c, a.ys, a.c4y, a.s4y, j, c5, rik, fu, fv);
      acoustic_F<T, MAT>(dxp, dyp, dxu, dyv, rik, Kk, fu, fv, K[0], K[1], K[2]);
      if (xe || yc) {  // boundary terms, as in edge_rhs
        const T qinv0 = T(Ops<ORDER>::hqinv[0]);
        const T hqx = a.hix * qinv0, hqy = a.hiy * qinv0;
        const int bc = a.bc == B_DEFAULT ? B_FSREF : a.bc;
        const T u = Yc[0], v = Yc[1], p = Yc[2];
        if (bc == B_FSREF) {
          if (gi == 0) K[0] -= hqx * p;
          if (gj == 0) K[1] -= hqy * p;
          if (gi == a.nx - 1) K[0] += hqx * p;
          if (gj == a.ny - 1) K[1] += hqy * p;
        } else if (bc == B_FS) {
          if (gi == 0) K[0] -= rik * (hqx * p);
          if (gj == 0) K[1] -= rik * (hqy * p);
          if (gi == a.nx - 1) K[0] += rik * (hqx * p);
          if (gj == a.ny - 1) K[1] += rik * (hqy * p);
        } else {
          if (gi == 0) K[2] -= Kk * (hqx * u);
          if (gj == 0) K[2] -= Kk * (hqy * v);
          if (gi == a.nx - 1) K[2] += Kk * (hqx * u);
          if (gj == a.ny - 1) K[2] += Kk * (hqy * v);
        }
      }
    } else {
      const T va = MAT == M_ARR ? rik : a.ax, vb = MAT == M_ARR ? Kk : a.ay;
      const T l = dlane(ax), w = drow(ay);
      T k = -mad(va, TR ? w : l, vb * (TR ? l : w));
      if (xe || yc) {
        const T qinv0 = T(Ops<ORDER>::hqinv[0]);
        const T hqx = a.hix * qinv0, hqy = a.hiy * qinv0, u = Yc[0];
        if (gi == 0) k += T(0.5) * (T(-0.5) * (va + fabs(va))) * (hqx * u);
        if (gj == 0) k += T(0.5) * (T(-0.5) * (vb + fabs(vb))) * (hqy * u);
        if (gi == a.nx - 1) k += T(0.5) * (T(0.5) * (va - fabs(va))) * (hqx * u);
        if (gj == a.ny - 1) k += T(0.5) * (T(0.5) * (vb - fabs(vb))) * (hqy * u);
      }
      K[0] = k;
    }
  }
};

// The RK4 step of a patch.
template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN, bool TR, int NW, int H>
__device__ __forceinline__ void step_patch(const StepArgs<T> &a, T *s_, int i0, int i1, int j0, int j1)
{
  using Pt = Patch<T, ORDER, PHYS, MAT, TR, NW, H, 4>;
  constexpr int KR = Pt::KR, C = Pt::C;
  constexpr bool AC = Pt::AC;
  const Pt pt(a, s_, i0, i1, j0, j1);

  T U[KR][C], P[KR][C], Y[KR][C], ri[KR], Kb[KR], cmp[KR][C];
#pragma unroll
  for (int k = 0; k < KR; k++) {
    const long o = pt.at(pt.row(k));
#pragma unroll
    for (int c = 0; c < C; c++) U[k][c] = a.u[c * a.plane + o];
    ri[k] = Kb[k] = T(1);
    if constexpr (MAT == M_ARR) {
      ri[k] = (AC ? a.rinv : a.velx)[o];
      Kb[k] = (AC ? a.bulk : a.vely)[o];
    }
    if constexpr (KAHAN) {
#pragma unroll
      for (int c = 0; c < C; c++) cmp[k][c] = a.comp[c * a.plane + o];
    }
  }
#pragma unroll
  for (int k = 0; k < KR; k++)
#pragma unroll
    for (int c = 0; c < C; c++) {
      Y[k][c] = U[k][c];
      P[k][c] = T(0);
      pt.slot(0, pt.wv + NW * k)[c * Pt::FS] = U[k][c];
    }
  __syncthreads();

  // (unrolled: fewer registers, so two blocks per CU; 513^2 18.9 against 27 us)
  auto stages = [&](auto XE) {
#pragma unroll
    for (int st = 1; st <= 4; st++) {
      const int b = (st - 1) & 1;
      const double c5 = st == 1 ? a.c5[0] : (st == 4 ? a.c5[2] : a.c5[1]);
      const T cy = st == 3 ? a.c3 : a.c12, w = st == 2 ? T(2) : T(1);
#pragma unroll
      for (int k = 0; k < KR; k++) {
        const int r = pt.wv + NW * k, j = pt.yl[0] + r;
        if (j < pt.yl[st] || j >= pt.yh[st]) continue;  // (the whole wave)
        T K[C];
        pt.template rhs<decltype(XE)::value>(b, r, j, Y[k], ri[k], Kb[k], c5, K);
        if (st < 4) {
#pragma unroll
          for (int c = 0; c < C; c++) {
            const T y = mad(cy, K[c], U[k][c]);
            P[k][c] = P[k][c] + w * (y - U[k][c]);  // exact products: Y2-U, + 2 (Y3-U), + (Y4-U)
            Y[k][c] = y;
            pt.slot(b ^ 1, r)[c * Pt::FS] = y;
          }
        } else if (pt.own()) {
          const long o = pt.at(j);
#pragma unroll
          for (int c = 0; c < C; c++) {
            const T inc = mad(P[k][c], a.third, a.ca * K[c]);
            if constexpr (!KAHAN) {
              a.uo[c * a.plane + o] = U[k][c] + inc;
            } else {
              const T y = inc - cmp[k][c];
              const T t = U[k][c] + y;
              a.comp[c * a.plane + o] = (t - U[k][c]) - y;
              a.uo[c * a.plane + o] = t;
            }
          }
        }
      }
      __syncthreads();
    }
  };
  if (!TR && pt.xedge) stages(std::integral_constant<bool, !TR>{});
  else stages(std::false_type{});
}

template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN>
__global__ __launch_bounds__(64 * kStepWaves) void step2d_kernel(StepArgs<T> a)
{
  constexpr int H = kStepWaves * step_rows(ORDER);
  __shared__ T s[step_lds(ORDER, PHYS == PH_ACOUSTIC ? 3 : 1, H)];
  const int i0 = (blockIdx.x % a.px) * a.pw, j0 = (blockIdx.x / a.px) * a.ph;
  step_patch<T, ORDER, PHYS, MAT, KAHAN, false, kStepWaves, H>(a, s, i0, min(i0 + a.pw, a.nx), j0,
                                                               min(j0 + a.ph, a.ny));
}

// The cut of an nx x ny grid into patches; ok: every region fits a block.
// Patches are as low as gives each a CU of its own, since a block's time is
// its rows' (101^2, order 4: 7.4 us per step at 2 rows, 9.0 at 8), and as high
// as the rows of a block allow on grids that fill the chip anyway (513^2: 18.9
// us at 8 rows, 22.5 at 4).
struct StepPlan {
  bool ok;
  int px, pw, py, ph;
};
// stages of the method, most rows a block loads, least and most rows of a patch
template <int ORDER> inline StepPlan patch_plan(int nx, int ny, int stages, int rows, int least, int most)
{
  // parts of `len` points of a line of n whose regions hold at most `cap`
  auto fits = [=](int n, int len, int cap) {
    for (int p = 0; p < n; p += len) {
      int lo = p, hi = p + len < n ? p + len : n;
      for (int k = 0; k < stages; k++) stencil_reach<ORDER>(lo, hi, n);
      if (hi - lo > cap) return false;
    }
    return true;
  };
  StepPlan p{};
  p.px = (nx + kStepLanes - 1) / kStepLanes;
  for (;; p.px++) {
    p.pw = (nx + p.px - 1) / p.px;
    if (p.pw < 1 || fits(nx, p.pw, kStepLanes)) break;
    if (p.pw == 1) return p;
  }
  p.px = (nx + p.pw - 1) / p.pw;
  constexpr int kCus = 256;
  int best = 0;
  for (p.ph = least; p.ph <= most; p.ph++) {
    if (!fits(ny, p.ph, rows)) continue;
    best = p.ph;
    if ((long)p.px * ((ny + p.ph - 1) / p.ph) <= kCus) break;
  }
  if (!best) return p;
  p.ph = best;
  p.py = (ny + p.ph - 1) / p.ph;
  p.ok = true;
  return p;
}
template <int ORDER> inline StepPlan step_plan_t(int nx, int ny)
{
  return patch_plan<ORDER>(nx, ny, 4, kStepWaves * step_rows(ORDER), 1, 8);
}
inline StepPlan step_plan(int order, int nx, int ny)
{
  return order == 2 ? step_plan_t<2>(nx, ny) : (order == 4 ? step_plan_t<4>(nx, ny) : step_plan_t<6>(nx, ny));
}

// Marched steps (sbp_march.hpp): output columns of a strip, depth of the frame
// around the strips, the frame's patches (px along the bottom and top each,
// one per kStepLanes - 4 order rows at either side).
constexpr int kMarchThreads = 256;
constexpr int march_cols(int order) { return kMarchThreads - 4 * order; }
constexpr int march_depth(int order) { return order == 2 ? 4 : (order == 4 ? 10 : 15); }
constexpr int step_cols(int order) { return kStepLanes - 4 * order; }
__host__ __device__ inline int march_frame(int order, int px, int ny)
{
  return 2 * px + 2 * ((ny - 2 * march_depth(order) + step_cols(order) - 1) / step_cols(order));
}

// The cut of the marched region into strips and segments.  A segment costs its
// rows and the 4 order rows it leads in with, and each further block per CU
// slows the others down by about a quarter of what one alone takes (4097^2
// FP32 172 / 122 / 126 / 116 us per step at 1 .. 4 per CU, 2049^2 51 / 38 / 38
// / 38, 1025^2 21 / 19 / 18 / 21): as many blocks per CU, at most `resident`,
// as make (rows + lead) (1 + w / 4) smallest.  A frame of few patches takes
// its place within them, so that all blocks of a launch run at once (1025^2
// FP64: 28.5 us per step, 31.7 with another 88 blocks to wait for); a larger one
// is worth a longer launch (4097^2 FP64 216 / 302).  Where a
// CU holds one block (order 6 FP64) patches that follow wait for whole blocks
// and cost about as much as 3 order rows, so the cheaper of the two is taken,
// rows counted as they run, in whole groups of order + 1 (us per step, within /
// after the strips' blocks: 1133 x 132 22 / 36, 1395 x 129 23 / 36, 500 x 800 29
// / 42; 3428 x 140 43 / 38, 1111 x 1053 with arrays 65 / 61).
struct MarchPlan {
  bool ok;
  int strips, segs, seg_rows;
};
inline MarchPlan march_plan(int order, int nx, int ny, int px, int resident)
{
  constexpr int kCus = 256;
  const int D = march_depth(order), w = nx - 2 * D, h = ny - 2 * D;
  MarchPlan p{};
  if (w < 1 || h < 1 || px < 1 || resident < 1) return p;
  p.strips = (w + march_cols(order) - 1) / march_cols(order);
  const int nf = march_frame(order, px, ny);
  double least = 1e300;
  auto consider = [&](int per, int blocks, int group, int late) {
    const int segs = blocks > p.strips ? blocks / p.strips : 1;
    const int rows = (h + segs - 1) / segs;
    const double cost = ((rows + group - 1) / group * group + 4.0 * order + late) * (4 + per);
    if (cost < least) {
      least = cost;
      p.seg_rows = rows;
    }
  };
  for (int per = 1; per <= resident; per++) {
    const int all = kCus * per;
    if (resident > 1) {
      consider(per, 4 * nf <= all ? all - nf : all, 1, 0);
    } else {
      if (all - nf >= p.strips) consider(per, all - nf, order + 1, 0);
      consider(per, all, order + 1, 3 * order);
    }
  }
  p.segs = (h + p.seg_rows - 1) / p.seg_rows;
  p.ok = true;
  return p;
}

template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN> struct StepLauncher {
  static hipError_t launch(const void *args, int grid, hipStream_t s)
  {
    hipLaunchKernelGGL((step2d_kernel<T, ORDER, PHYS, MAT, KAHAN>), dim3(grid), dim3(64 * kStepWaves), 0, s,
                       *static_cast<const StepArgs<T> *>(args));
    return hipGetLastError();
  }
};

}  // namespace sbp
