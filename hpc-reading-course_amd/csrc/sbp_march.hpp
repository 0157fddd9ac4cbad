// sbp_march.hpp -- a whole RK4 step of a large 2D grid in one pass over memory.
//
// A block of NT threads owns NT columns (NT - 8R of them outputs), one per
// thread, and marches down a segment of rows.  Iteration k takes row r = j0 -
// 4R + k of U; stage s of the step (1 .. 4) is evaluated at row r - sR from
// the rows the stage before it has produced, so U is read once and U' written
// once per step (2 words per value instead of the 5 of two launches).  Each
// thread keeps the last 2R+1 rows of every stage's operand of its own column
// in registers: the y stencils, centre values and the RK4 combination come
// from there.  The x neighbours come from LDS, to which every operand row is
// written as it is formed; a row becomes the centre of its stage's stencils R
// iterations later, so a ring of R+1 rows needs one barrier per iteration and
// no value is waited for across it.  The register rings have 2R+1 slots and
// the row loop is unrolled 2R+1 times, so a slot is a fixed register and rows
// move by renaming:
//   U1   rows r .. r-2R of U        U2   rows r-2R-1 .. r-4R (stages 3 and 4)
//   Y2, Y3, Y4  the last 2R+1 rows of each stage's result
//   S    (Y2-U) + 2 (Y3-U) [+ (Y4-U)] of rows r-2R .. r-4R
// The arithmetic per point is that of the other schedules, term for term.
//
// The strips cover [D, nx-D) x [D, ny-D) with D = CLS + 3R, so every point of
// every stage is an interior point of the operator; the D-deep frame is cut
// into patches that blocks of the same launch step on chip (sbp_step.hpp).
//
// What bounds it: order 4 FP64, 4097^2, takes 217 us per step (452 as two
// launches).  806 MB of U and U' are 147 us at what a copy reaches; a row costs
// a CU's LDS 0.6 us for the neighbours (32 words read and 8 written per column)
// and its SIMDs 0.8 us for 200 instructions, which the barrier of each row lets
// overlap in part; halo columns and lead-in rows add a fifth.  Constant LDS
// addresses (15 instructions less per row, at a longer unrolling) and more rows
// of loads in flight (3, 4) gain nothing.  Small grids wait for the lead-in
// and the frame (1025^2 26 us, 47.5 before).  FP32 4097^2 116 (236), order 6
// FP32 + compensation with rho/K arrays 273 (442), order 6 FP64 347 (570: its
// rings fill the register file, one wave per SIMD).  Stores are cached: 2049^2
// FP64 74.6 us, 78.5 nontemporal, and the next step reads them.  A version
// whose waves exchange columns through DPP alone, with no LDS and no barrier,
// needs 64 - 8R output columns per wave: 255 and FP32 139 us at 4097^2.
#pragma once
#include <utility>

#include "sbp_batch.hpp"
#include "sbp_step.hpp"

namespace sbp {

template <int V> struct Int {
  static constexpr int value = V;
};
template <class F, int... K> __device__ __forceinline__ void each_int(F &f, std::integer_sequence<int, K...>)
{
  (f(Int<K>{}), ...);
}

// A ring of WN rows of N values per thread: registers, or (LDS) memory of the
// thread's own, slots being compile-time constants either way.
template <typename T, int WN, int N, bool LDS> struct LaneRing {
  T v[WN][N];
  __device__ __forceinline__ explicit LaneRing(T *) {}
  template <int S> __device__ __forceinline__ T get(int c) const { return v[S][c]; }
  template <int S> __device__ __forceinline__ void set(int c, T x) { v[S][c] = x; }
};
// (volatile: the compiler would otherwise keep every row in registers too)
template <typename T, int WN, int N> struct LaneRing<T, WN, N, true> {
  typedef __attribute__((address_space(3))) T LT;
  LT *p;
  __device__ __forceinline__ explicit LaneRing(T *base) : p((LT *)base) {}
  template <int S> __device__ __forceinline__ T get(int c) const
  {
    return *const_cast<const volatile LT *>(p + (S * N + c) * kMarchThreads);
  }
  template <int S> __device__ __forceinline__ void set(int c, T x) { p[(S * N + c) * kMarchThreads] = x; }
};

// Whether the ring S lives in LDS: where FP64 acoustics would need more than
// 256 registers with it, two waves per SIMD (order 4 with arrays; 39 us per step
// at 1025^2 in registers, 33 in LDS) or all the more of the second half of the
// file (order 6).  LDS is the scarcer where they suffice: order 4 without
// arrays 27.1 / 30.2 us at 1025^2, 67 / 74 at 2049^2, 226 / 236 at 4097^2.
constexpr bool march_s_lds(int esz, int order, bool acoustic, bool arrays)
{
  return esz == 8 && acoustic && (order == 6 || (order == 4 && arrays));
}
// LDS values per block of that ring, and of the exchanged rows: R+1 slots of
// the differentiated fields of the four operands, R columns beyond either end
constexpr int march_ring(int order, int comps) { return comps * (order + 1) * kMarchThreads; }
constexpr int march_rows(int order, int comps)
{
  return (order / 2 + 1) * 4 * (comps == 3 ? 2 : 1) * (kMarchThreads + order);
}

template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN>
__device__ __forceinline__ void march_strip(const StepArgs<T> &a, T *lds, int strip, int j0, int j1)
{
  using O = Ops<ORDER>;
  constexpr int R = O::R, WN = 2 * R + 1, D = march_depth(ORDER), PF = 2, NT = kMarchThreads;
  constexpr bool AC = PHYS == PH_ACOUSTIC, LD_M = MAT == M_ARR;
  constexpr int C = AC ? 3 : 1, NF = AC ? 2 : 1;
  constexpr int XW = NT + 2 * R, XS = 4 * NF * XW;  // an exchanged row, a slot of them
  static_assert(D == O::CLS + 3 * R && MAT != M_REF, "marched region");

  const int t = threadIdx.x;
  const int i = D + strip * march_cols(ORDER) - 4 * R + t;
  const int ic = a.xoff + min(i, a.nx - 1);
  const bool out = t >= 4 * R && t < NT - 4 * R && i < a.nx - D;
  const int jmax = a.ny - 1, rs = j0 - 4 * R;
  T *const x = lds + R + t;  // this thread's column of the exchanged rows

  T U1[WN][C], U2[WN][C], Y2[WN][C], Y3[WN][C], Y4[WN][C], q[WN][C];
  LaneRing<T, WN, C, march_s_lds(sizeof(T), ORDER, AC, LD_M)> S(lds + march_rows(ORDER, C) + t);
  // materials (or velocities) of rows r-R .. r-3R, and of r-3R .. r-4R
  T M1[WN][2], M2[WN][2];
  T qr[WN], qk[WN], qc[WN][C];

  // row k of U, material row k - R, compensation row k - 4R -> slot
  auto load = [&](int k, int slot) {
    const T *__restrict__ p = a.u + (long)min(rs + k, jmax) * a.pitch;
#pragma unroll
    for (int c = 0; c < C; c++) q[slot][c] = p[c * a.plane + ic];
    if constexpr (LD_M) {
      const long o = (long)max(min(rs + k, jmax) - R, 0) * a.pitch;
      qr[slot] = (AC ? a.rinv : a.velx)[o + ic];
      qk[slot] = (AC ? a.bulk : a.vely)[o + ic];
    }
    if constexpr (KAHAN) {
      const T *__restrict__ pc = a.comp + (long)max(min(rs + k, jmax) - 4 * R, 0) * a.pitch;
#pragma unroll
      for (int c = 0; c < C; c++) qc[slot][c] = ldg<true>(pc + c * a.plane + ic);
    }
  };

  // x neighbours of one exchanged field (unit: stage and field) of the row at xr
  auto fetch = [&](int unit, const T *xr, T (&o)[2 * R]) {
    const T *l = xr + unit * XW;
#pragma unroll
    for (int n = 0; n < 2 * R; n++) o[n] = l[n < R ? n - R : n - R + 1];
  };
  // right-hand side of stage ST (of NS running) at ring slot s of its operand
  // rows Y, whose centre row lies in the exchange slot at xr.  The neighbours of
  // a field are fetched while the field before it is differentiated, behind a
  // scheduling barrier: left to itself the compiler moves each fetch to its use
  // and waits for LDS eight times per row (order 6 FP64, one wave per SIMD, 413
  // us per step at 4097^2, 347 so; order 4 FP64 27.2 and 26.3 at 1025^2).  A
  // whole stage ahead would take order 4 FP64 past 256 registers.
  auto rhs = [&](const T (&Y)[WN][C], auto SLOT, auto ST, auto NS, T (&nb)[2][2 * R], const T *xr, T ri, T Kb, T *F) {
    constexpr int s = decltype(SLOT)::value, st = decltype(ST)::value - 1, units = decltype(NS)::value * NF;
    auto ddx = [&](auto FIELD, int c) {
      constexpr int u = st * NF + decltype(FIELD)::value;
      if constexpr (u + 1 < units) fetch(u + 1, xr, nb[(u + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const T (&l)[2 * R] = nb[u & 1];
      return dint<T, ORDER>([&](int n) { return n == R ? Y[s][c] : l[n < R ? n : n - 1]; }, a.hix);
    };
    auto ddy = [&](int c) { return dint<T, ORDER>([&](int n) { return Y[(s + n + WN - R) % WN][c]; }, a.hiy); };
    if constexpr (AC) {
      const T dxu = ddx(Int<0>{}, 0), dyv = ddy(1), dxp = ddx(Int<1>{}, 2), dyp = ddy(2);
      acoustic_F<T, MAT>(dxp, dyp, dxu, dyv, ri, Kb, T(0), T(0), F[0], F[1], F[2]);
    } else {
      const T va = LD_M ? ri : a.ax, vb = LD_M ? Kb : a.ay;
      F[0] = -mad(va, ddx(Int<0>{}, 0), vb * ddy(0));
    }
  };
  // a new operand row of stage ST into the exchange slot at xw
  auto share = [&](auto ST, T *xw, const T *Y) {
    constexpr int st = decltype(ST)::value - 1;
    xw[st * NF * XW] = Y[0];
    if constexpr (AC) xw[(st * NF + 1) * XW] = Y[2];
  };

  // iteration k (ring slot KP = k mod WN) with the first NS stages running
  int slot = 0;  // k mod (R + 1): the exchange slot written
  auto iter = [&](auto KP, auto NS, int k) {
    constexpr int kp = decltype(KP)::value, ns = decltype(NS)::value;
    constexpr int s1 = (kp + 2 * WN - R) % WN, s2 = (kp + 2 * WN - 2 * R) % WN, s3 = (kp + 4 * WN - 3 * R) % WN,
                  s4 = (kp + 4 * WN - 4 * R) % WN;
    T *const xw = x + slot * XS;
    slot = slot == R ? 0 : slot + 1;
    const T *const xr = x + slot * XS;  // written R iterations ago
    T Cm[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
      U2[kp][c] = U1[kp][c];
      U1[kp][c] = q[kp][c];
      if constexpr (KAHAN) Cm[c] = qc[kp][c];
    }
    share(Int<1>{}, xw, U1[kp]);
    const T mr = LD_M ? qr[kp] : T(1), mk = LD_M ? qk[kp] : T(1);
    if constexpr (LD_M) {
      M1[s1][0] = mr;
      M1[s1][1] = mk;
    }
    load(k + PF, (kp + PF) % WN);
    T F[C], nb[2][2 * R];
    if constexpr (ns >= 1) {
      fetch(0, xr, nb[0]);
      rhs(U1, Int<s1>{}, Int<1>{}, NS, nb, xr, mr, mk, F);
#pragma unroll
      for (int c = 0; c < C; c++) Y2[s1][c] = mad(a.c12, F[c], U1[s1][c]);
      share(Int<2>{}, xw, Y2[s1]);
    }
    if constexpr (ns >= 2) {
      rhs(Y2, Int<s2>{}, Int<2>{}, NS, nb, xr, LD_M ? M1[s2][0] : T(1), LD_M ? M1[s2][1] : T(1), F);
#pragma unroll
      for (int c = 0; c < C; c++) {
        const T U = U1[s2][c];
        Y3[s2][c] = mad(a.c12, F[c], U);
        S.template set<s2>(c, (Y2[s2][c] - U) + 2 * (Y3[s2][c] - U));
      }
      share(Int<3>{}, xw, Y3[s2]);
    }
    if constexpr (ns >= 3) {
      const T m3r = LD_M ? M1[s3][0] : T(1), m3k = LD_M ? M1[s3][1] : T(1);
      if constexpr (LD_M) {
        M2[s3][0] = m3r;
        M2[s3][1] = m3k;
      }
      rhs(Y3, Int<s3>{}, Int<3>{}, NS, nb, xr, m3r, m3k, F);
#pragma unroll
      for (int c = 0; c < C; c++) {
        const T U = U2[s3][c];
        Y4[s3][c] = mad(a.c3, F[c], U);
        S.template set<s3>(c, S.template get<s3>(c) + (Y4[s3][c] - U));
      }
      share(Int<4>{}, xw, Y4[s3]);
    }
    if constexpr (ns >= 4) {
      rhs(Y4, Int<s4>{}, Int<4>{}, NS, nb, xr, LD_M ? M2[s4][0] : T(1), LD_M ? M2[s4][1] : T(1), F);
      const long o = (long)(rs + k - 4 * R) * a.pitch;
      if (out && rs + k - 4 * R < j1) {
        T *__restrict__ p = a.uo + o;
#pragma unroll
        for (int c = 0; c < C; c++) {
          const T U = U2[s4][c], inc = mad(S.template get<s4>(c), a.third, a.ca * F[c]);
          if constexpr (!KAHAN) {
            stg<false>(p + c * a.plane + ic, U + inc);
          } else {
            const T y = inc - Cm[c];
            const T w = U + y;
            stg<false>(a.comp + o + c * a.plane + ic, (w - U) - y);
            stg<false>(p + c * a.plane + ic, w);
          }
        }
      }
    }
    __syncthreads();
  };

#pragma unroll
  for (int k = 0; k < PF; k++) load(k, k % WN);
  // the first rows: 2R of U alone, then each further stage after 2R more
  auto lead = [&](auto K) {
    constexpr int kk = decltype(K)::value;
    iter(Int<kk % WN>{}, Int<kk / (2 * R)>{}, kk);
  };
  each_int(lead, std::make_integer_sequence<int, 8 * R>{});
  // (a segment has at least one row; a loop that might not run would let the
  // compiler sink the leading rows' results into it, with all their operands.
  // Rows run in whole groups of 2R+1: the last group's surplus is computed and
  // dropped, so 12 rows of order 4 cost 15)
  const int nk = (j1 - j0) + 8 * R;
  int k = 8 * R;
  auto row = [&](auto N) { iter(Int<(8 * R + decltype(N)::value) % WN>{}, Int<4>{}, k + decltype(N)::value); };
  do {
    each_int(row, std::make_integer_sequence<int, WN>{});
    k += WN;
  } while (k < nk);
}

// rows a frame patch loads: D and what four stages reach on one side, in whole rows of the block's waves
constexpr int march_frame_rows(int order)
{
  return (march_depth(order) + 2 * order + kMarchThreads / 64 - 1) / (kMarchThreads / 64) * (kMarchThreads / 64);
}

// block b's frame patch
template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN>
__device__ __forceinline__ void march_frame_patch(const StepArgs<T> &a, T *s, int b)
{
  constexpr int D = march_depth(ORDER), LEN = step_cols(ORDER), NW = kMarchThreads / 64, H = march_frame_rows(ORDER);
  if (b < 2 * a.px) {
    const int i0 = (b % a.px) * a.pw, j0 = b < a.px ? 0 : a.ny - D;
    step_patch<T, ORDER, PHYS, MAT, KAHAN, false, NW, H>(a, s, i0, min(i0 + a.pw, a.nx), j0, j0 + D);
  } else {
    b -= 2 * a.px;
    const int j0 = D + (b >> 1) * LEN, i0 = b & 1 ? a.nx - D : 0;
    step_patch<T, ORDER, PHYS, MAT, KAHAN, true, NW, H>(a, s, j0, min(j0 + LEN, a.ny - D), i0, i0 + D);
  }
}

// values of a block's LDS: a marching block's, or a frame patch's
template <typename T> constexpr int march_block_lds(int order, int comps, bool arrays)
{
  const int m =
      march_rows(order, comps) + (march_s_lds(sizeof(T), order, comps == 3, arrays) ? march_ring(order, comps) : 0);
  const int f = step_lds(order, comps, march_frame_rows(order));
  return m > f ? m : f;
}

template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN>
__global__ __launch_bounds__(kMarchThreads) void march2d_kernel(StepArgs<T> a, int frame)
{
  constexpr int D = march_depth(ORDER), NC = PHYS == PH_ACOUSTIC ? 3 : 1;
  __shared__ T lds[march_block_lds<T>(ORDER, NC, MAT == M_ARR)];
  if ((int)blockIdx.x < frame) {
    march_frame_patch<T, ORDER, PHYS, MAT, KAHAN>(a, lds, blockIdx.x);
    return;
  }
  // every XCD takes a contiguous run of tiles (strips of one segment after
  // another): neighbouring strips share halo columns, segments halo rows
  const int nb = gridDim.x - frame, b = blockIdx.x - frame, xcd = b % kNumXcd, local = b / kNumXcd;
  const int q = nb / kNumXcd, r = nb % kNumXcd;
  const int w = xcd * q + min(xcd, r) + local;
  const int strip = w % a.strips, seg = w / a.strips;
  const int j0 = D + seg * a.seg_rows, j1 = min(j0 + a.seg_rows, a.ny - D);
  march_strip<T, ORDER, PHYS, MAT, KAHAN>(a, lds, strip, j0, j1);
}

template <typename T, int ORDER, int PHYS, int MAT, bool KAHAN> struct MarchLauncher {
  static hipError_t launch(const void *args, hipStream_t s)
  {
    const StepArgs<T> &a = *static_cast<const StepArgs<T> *>(args);
    const int nf = march_frame(ORDER, a.px, a.ny);
    hipLaunchKernelGGL((march2d_kernel<T, ORDER, PHYS, MAT, KAHAN>), dim3(nf + a.strips * a.segs), dim3(kMarchThreads), 0,
                       s, a, nf);
    return hipGetLastError();
  }
  // blocks a CU holds
  static hipError_t resident(int *blocks)
  {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, march2d_kernel<T, ORDER, PHYS, MAT, KAHAN>,
                                                        kMarchThreads, 0);
  }
  static MarchFns fns() { return {&launch, &resident}; }
};

template <typename T, int ORDER, bool KAHAN> MarchFns pick_march(int phys, int mat)
{
  if (phys == PH_ACOUSTIC && mat == M_UNIT) return MarchLauncher<T, ORDER, PH_ACOUSTIC, M_UNIT, KAHAN>::fns();
  if (phys == PH_ACOUSTIC && mat == M_ARR) return MarchLauncher<T, ORDER, PH_ACOUSTIC, M_ARR, KAHAN>::fns();
  if (phys == PH_ADV2D && mat == M_UNIT) return MarchLauncher<T, ORDER, PH_ADV2D, M_UNIT, KAHAN>::fns();
  if (phys == PH_ADV2D && mat == M_ARR) return MarchLauncher<T, ORDER, PH_ADV2D, M_ARR, KAHAN>::fns();
  return {};
}

// --------------------------------------------------------------------------
// Ensembles: one launch steps every instance, a block per item of the work
// list (laid out as in sbp_batch.hpp: a chunk per XCD, whose blocks take its
// items in order), segments first and then the frames' patches.  FP32, 48
// instances of 129^2 .. 1025^2 with rho/K arrays, order 4: 421 us per step in
// two launches, 199 marched; 16 of 257^2 37 and 25.  A block per item, not persistent blocks: the
// items' sizes differ by a factor of ten and the hardware hands them out.
// --------------------------------------------------------------------------
template <typename T, int ORDER, int MAT, bool KAHAN>
__global__ __launch_bounds__(kMarchThreads) void batch_march_kernel(const BatchInst<T> *__restrict__ inst,
                                                                   const int2 *__restrict__ work)
{
  constexpr int D = march_depth(ORDER);
  __shared__ T lds[march_block_lds<T>(ORDER, 3, MAT == M_ARR)];
  const int2 chunk = work[blockIdx.x % kNumXcd];
  const int w = blockIdx.x / kNumXcd;
  if (w >= chunk.y) return;
  const int2 it = work[kNumXcd + chunk.x + w];
  const BatchInst<T> &d = inst[it.x];
  StepArgs<T> a{};
  a.u = d.U;
  a.uo = d.Y0;
  a.comp = d.comp;
  a.rinv = d.rinv;
  a.bulk = d.bulk;
  a.plane = d.plane;
  a.pitch = d.pitch;
  a.xoff = d.xoff;
  a.nx = d.nx;
  a.ny = d.ny;
  a.bc = d.bc;
  a.hix = d.hix;
  a.hiy = d.hiy;
  const double dt = d.dt;
  a.c12 = T(0.5 * dt);
  a.c3 = T(dt);
  a.ca = T(dt / 6);
  a.third = T(1.0 / 3.0);
  a.px = d.m_px;
  a.pw = d.m_pw;
  if (it.y < d.m_frame) {
    march_frame_patch<T, ORDER, PH_ACOUSTIC, MAT, KAHAN>(a, lds, it.y);
    return;
  }
  const int t = it.y - d.m_frame, strip = t % d.m_strips;
  const int j0 = D + t / d.m_strips * d.m_seg_rows, j1 = min(j0 + d.m_seg_rows, d.ny - D);
  march_strip<T, ORDER, PH_ACOUSTIC, MAT, KAHAN>(a, lds, strip, j0, j1);
}

template <typename T, int ORDER, int MAT, bool KAHAN> struct BatchMarchLauncher {
  static hipError_t launch(int, const void *inst, const int2 *work, int, int grid, hipStream_t s)
  {
    hipLaunchKernelGGL((batch_march_kernel<T, ORDER, MAT, KAHAN>), dim3(grid), dim3(kMarchThreads), 0, s,
                       static_cast<const BatchInst<T> *>(inst), work);
    return hipGetLastError();
  }
};

template <typename T, int ORDER, bool KAHAN> BatchLaunchFn pick_batch_march(int mat)
{
  return mat == M_ARR ? &BatchMarchLauncher<T, ORDER, M_ARR, KAHAN>::launch
                      : &BatchMarchLauncher<T, ORDER, M_UNIT, KAHAN>::launch;
}

}  // namespace sbp
