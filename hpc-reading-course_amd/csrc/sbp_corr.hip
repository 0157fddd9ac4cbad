// sbp_corr.hip -- learned coarse-grid corrector: a 3-layer 3x3 convolutional
// network (8 -> 32 -> 32 -> 3 channels, ReLU) applied to the state after each
// coarse RK4 step.  Its inputs at each point are eight normalised features of
// the state and the materials (the fourth-difference terms of the stencil's
// leading truncation error, the fourth differences of u, v and p, rho and
// K: pack_state_tiled_kernel / pack_batch_tiled_kernel below).  Every
// convolution and gradient runs on v_mfma_f32_16x16x32_bf16 with FP32
// accumulation; master weights and Adam moments are FP32.  No counterpart in the
// reference: the plain fine-grid solve of the same path is its fallback and
// reference, and a correction that lifts the discrete energy above the
// energy the solve started from by more than a set bound is rejected.
//
// Activations are channels-last [image][y][x][channel] in bf16.  Forward
// (fused_net_kernel, inference and training) and backward-data
// (fused_back_kernel) march down windows of an image with all layers in one
// kernel; weight gradients (wgrad_kernel) are GEMMs reduced over pixels,
// written as per-block partials and summed in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/sbp_hip.h"
#include "sbp_batch_impl.hpp"
#include "sbp_corr_plan.hpp"
#include "sbp_ctx.hpp"
#include "sbp_host.hpp"

using namespace sbp;
using sbp::host::fail;
#define HIP_OR_FAIL(expr) SBP_HIP_OR_FAIL(expr)

namespace {

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef unsigned short bf16;

// Network shape.
constexpr int C_IN = 8, C_INP = 8, C_H = 32, C_OUT = 3, C_OUTP = 16;
// normalisation block: shift[C_IN], scale[C_IN], out_scale[C_OUT]
constexpr int NORM_OUT = 2 * C_IN, NORM_LEN = 2 * C_IN + C_OUT;
constexpr int KP1 = 80;   // 9*8 = 72 padded to 80
constexpr int KP2 = 288;  // 9*32
constexpr int KP3 = 288;
constexpr int C_D3 = 8;   // channels of the output gradient in memory (3 real); its transposed weights take KP1
constexpr int N_W1 = C_H * C_IN * 9, N_B1 = C_H;
constexpr int N_W2 = C_H * C_H * 9, N_B2 = C_H;
constexpr int N_W3 = C_OUT * C_H * 9, N_B3 = C_OUT;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + N_W1, OFF_W2 = OFF_B1 + N_B1, OFF_B2 = OFF_W2 + N_W2;
constexpr int OFF_W3 = OFF_B2 + N_B2, OFF_B3 = OFF_W3 + N_W3, N_PARAMS = OFF_B3 + N_B3;

__device__ __forceinline__ bf16 f2bf(float f)
{
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16)((u >> 16) | 0x40u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (bf16)(u >> 16);
}

// Whether the correction acts at grid point (i, j) of an H x W image: the
// points closer than `band` to a wall (the boundary-closure rows) keep the
// plain scheme's values, and the training loss ignores them.
__device__ __forceinline__ bool corrected_at(int i, int j, int W, int H, int band)
{
  return min(min(i, W - 1 - i), min(j, H - 1 - j)) >= band;
}

// MSE loss over the C_OUT real channels and its gradient 2(y - t)/N in bf16
// (C_D3 channels per pixel; the padded channels, and points outside the
// corrected region, zero; N counts every point).  Per-block partial sums of
// squares in FP64.
__global__ __launch_bounds__(256) void loss_kernel(const float *__restrict__ y, const float *__restrict__ t, long npix,
                                                   int H, int W, int band, double inv_n, bf16 *__restrict__ dY,
                                                   double *__restrict__ partial)
{
  __shared__ double sh[256];
  double s = 0;
  const long npi = (long)H * W;
  for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += (long)gridDim.x * 256) {
    const long q = p % npi;
    const int j = (int)(q / W), i = (int)(q - (long)j * W);
    const bool on = corrected_at(i, j, W, H, band);
    __attribute__((aligned(16))) bf16 g[C_D3] = {0};
#pragma unroll
    for (int c = 0; c < C_OUT; c++) {
      const float d = y[p * C_OUT + c] - t[p * C_OUT + c];
      if (on) {
        s += (double)d * d;
        g[c] = f2bf((float)(2.0 * inv_n) * d);
      }
    }
    *reinterpret_cast<uint4 *>(dY + p * C_D3) = *reinterpret_cast<const uint4 *>(g);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// Adam on the FP32 master parameters.
__global__ __launch_bounds__(256) void adam_kernel(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                                                   const float *__restrict__ g, int n, float lr, float b1, float b2,
                                                   float eps, float c1, float c2)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Master parameters -> padded bf16 weights (forward and mirrored-transposed
// backward-data copies) and FP32 padded biases.
__global__ __launch_bounds__(256) void prepare_weights_kernel(const float *__restrict__ p, bf16 *__restrict__ w1,
                                                              bf16 *__restrict__ w2, bf16 *__restrict__ w3,
                                                              bf16 *__restrict__ w2t, bf16 *__restrict__ w3t,
                                                              float *__restrict__ b1, float *__restrict__ b2,
                                                              float *__restrict__ b3)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  // forward layer 1: [32][80]
  if (i < C_H * KP1) {
    const int co = i / KP1, k = i % KP1, tap = k / C_INP, ci = k % C_INP;
    w1[i] = (tap < 9 && ci < C_IN) ? f2bf(p[OFF_W1 + (co * C_IN + ci) * 9 + tap]) : (bf16)0;
  }
  if (i < C_H * KP2) {
    const int co = i / KP2, k = i % KP2, tap = k / C_H, ci = k % C_H;
    w2[i] = f2bf(p[OFF_W2 + (co * C_H + ci) * 9 + tap]);
    // backward-data of layer 2: W2T[ci][tap'*32 + co] = W2[co][8-tap'][ci]
    const int ci2 = i / KP2, k2 = i % KP2, tp = k2 / C_H, co2 = k2 % C_H;
    w2t[i] = f2bf(p[OFF_W2 + (co2 * C_H + ci2) * 9 + (8 - tp)]);
  }
  if (i < C_OUTP * KP3) {
    const int co = i / KP3, k = i % KP3, tap = k / C_H, ci = k % C_H;
    w3[i] = co < C_OUT ? f2bf(p[OFF_W3 + (co * C_H + ci) * 9 + tap]) : (bf16)0;
  }
  if (i < C_H * KP1) {
    // backward-data of layer 3: W3T[ci][tap'*8 + co] = W3[co][8-tap'][ci]
    const int ci = i / KP1, k = i % KP1, tp = k / C_D3, co = k % C_D3;
    w3t[i] = (tp < 9 && co < C_OUT) ? f2bf(p[OFF_W3 + (co * C_H + ci) * 9 + (8 - tp)]) : (bf16)0;
  }
  if (i < C_H) {
    b1[i] = p[OFF_B1 + i];
    b2[i] = p[OFF_B2 + i];
  }
  if (i < C_OUTP) b3[i] = i < C_OUT ? p[OFF_B3 + i] : 0.f;
}

// Raw per-point inputs (C_IN floats) -> normalised bf16 features.
__global__ __launch_bounds__(256) void pack_raw_kernel(const float *__restrict__ raw, long npix,
                                                       const float *__restrict__ shift_scale, bf16 *__restrict__ X)
{
  const long p = blockIdx.x * 256L + threadIdx.x;
  if (p >= npix) return;
#pragma unroll
  for (int c = 0; c < C_INP; c++)
    X[p * C_INP + c] = c < C_IN ? f2bf((raw[p * C_IN + c] - shift_scale[c]) * shift_scale[C_IN + c]) : (bf16)0;
}

// --------------------------------------------------------------------------
// Fused inference: the three convolutions of one image window in one kernel,
// activations kept in LDS.  A block owns a window of FW = 64 columns (image
// columns c0 .. c0+63, c0 = strip * 58 - 3) and a chunk of at most
// FUSED_MAX_ROWS output rows y0 .. y1-1, and marches down the rows.  Row step t:
//   * stores input row y0-3+t into slot t % 2 of the input ring;
//   * layer 1 reads input row q = y0-4+t (slot (t+1) % 2, stored in step
//     t-1) ONCE and adds its three row taps to the partial sums of layer-1
//     rows q+1 (tap dy = 0), q (dy = 1) and q-1 (dy = 2); row q-1 is then
//     complete and goes (bias, ReLU, bf16) into slot t % 2 of ring 1;
//   * layer 2 does the same with layer-1 row y0-6+t (completing row y0-7+t
//     into ring 2), layer 3 with layer-2 row y0-8+t (completing output row
//     y0-9+t into an LDS staging area that is written out after the march).
// Each layer reads only what the previous step wrote, so two slots per ring
// and one barrier per step order everything, and every activation row is
// read from LDS once per layer instead of once per row tap.  The three
// partial rows of layers 1 and 2 are three accumulators whose roles rotate
// each step; the step loop is unrolled by six, so ring slots and roles are
// compile-time constants.  Layer 3 has 3 output channels: its MFMA rows are
// (channel c, row tap dy) = 4c + dy, so one MFMA per column tap covers all
// three row taps, and the running sum moves on by one row tap per step inside
// each lane's four accumulator registers.  The input rows are fetched two
// steps ahead, and no global store is issued during the march, so a step
// never waits for more than the load issued two steps earlier.
//
// The GEMMs run on v_mfma_f32_16x16x32_bf16 with the weights as the A operand
// (M = 16 output channels) and the activations as B (N = 16 pixels of a
// segment, K = 32: one column tap of 32 channels, or the three column taps of
// the 8 input channels plus 8 zeros); a lane then holds 4 consecutive
// channels of one pixel, stored to LDS as one 8-byte write.  Every layer is
// evaluated on all 64 window columns; a value at window column w is exact
// when its inputs at w-1..w+1 are, so the output is exact on w in [3, 60]: 58
// output columns per window.  Activations at positions outside the image are
// zero (the network's zero padding).
// --------------------------------------------------------------------------
using bf16x8 = __attribute__((ext_vector_type(8))) short;
using vbf8 = __attribute__((ext_vector_type(8))) __bf16;
using vbf2 = __attribute__((ext_vector_type(2))) __bf16;
using f32x2 = __attribute__((ext_vector_type(2))) float;
using vi16x2 = __attribute__((ext_vector_type(2))) short;
constexpr int FPX = FW + 2;            // pixels per LDS row (one zero pad each side)
constexpr int F1S = 40;                // LDS channel stride of the 32-channel rows (80 B)
constexpr int FIN_PARTS = FPX * C_INP / 4;  // 8-byte parts of an input row

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vbf8, a), __builtin_bit_cast(vbf8, b), c, 0, 0, 0);
}

// 4 channels of one pixel (bias already in the sum): bf16 (round to nearest
// even), then ReLU as a signed 16-bit max with 0 (a bf16 is negative exactly
// when its sign bit is set, and -0 becomes +0 as the float ReLU makes it), or
// zero outside the image
__device__ __forceinline__ uint2 relu_pack4(f32x4 acc, bool in)
{
  const vi16x2 z = {0, 0};
  const vi16x2 lo = __builtin_elementwise_max(
      __builtin_bit_cast(vi16x2, __builtin_convertvector(f32x2{acc[0], acc[1]}, vbf2)), z);
  const vi16x2 hi = __builtin_elementwise_max(
      __builtin_bit_cast(vi16x2, __builtin_convertvector(f32x2{acc[2], acc[3]}, vbf2)), z);
  return uint2{in ? __builtin_bit_cast(unsigned, lo) : 0u, in ? __builtin_bit_cast(unsigned, hi) : 0u};
}

// The partial rows of layers 1 and 2 that one role holds (two segments each).
struct FusedRows {
  f32x4 l1[2], l2[2];
};

template <int V> using IC = std::integral_constant<int, V>;

// Energy of the corrected candidate, reduced in the inference kernel's
// epilogue (the batched corrected step): image k is the state of
// inst[k], and block b writes the H-weighted energy of U + out_scale * net
// over its output points to partial[b] (blocks of image k are contiguous).
struct NetEnergyArgs {
  const void *inst;  // BatchInst<T> of every image
  const float *out_scale;
  double *partial;
  int order, band;
};

// T: type of the state whose corrected energy the epilogue reduces; void for
// plain inference.  KEEP: also store the activations of layers 1 and 2 (the
// training forward; each block its own rows and 58 columns): 59 us for 16
// images of 257^2 against 289 us for one convolution launch per layer.
template <typename T, bool KEEP>
__global__ __launch_bounds__(256, 3) void fused_net_kernel(const bf16 *__restrict__ X, int nimg, int H, int W, int rows,
                                                        const bf16 *__restrict__ w1, const float *__restrict__ b1,
                                                        const bf16 *__restrict__ w2, const float *__restrict__ b2,
                                                        const bf16 *__restrict__ w3, const float *__restrict__ b3,
                                                        float *__restrict__ out, bf16 *__restrict__ keep1,
                                                        bf16 *__restrict__ keep2, NetEnergyArgs ea)
{
  __shared__ __attribute__((aligned(16))) bf16 s_in[2][FPX * C_INP];
  __shared__ __attribute__((aligned(16))) bf16 s_a1[2][FPX * F1S];
  __shared__ __attribute__((aligned(16))) bf16 s_a2[2][FPX * F1S];
  __shared__ float s_out[FUSED_MAX_ROWS * FOUT * C_OUT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kg = lane >> 4;
  const int strips = (W + FOUT - 1) / FOUT, chunks = (H + rows - 1) / rows;
  const int b = blockIdx.x;
  const int img = b / (strips * chunks), rem = b - img * strips * chunks;
  const int strip = rem / chunks, chunk = rem - strip * chunks;
  const int c0 = strip * FOUT - 3;  // image column of window column 0
  const int y0 = chunk * rows, y1 = min(y0 + rows, H);
  const long ibase = (long)img * H * W;

  // zero the activation rings once: the pad pixels stay zero
  for (int q = threadIdx.x; q < 2 * FPX * F1S; q += 256) {
    (&s_a1[0][0])[q] = 0;
    (&s_a2[0][0])[q] = 0;
  }

  // Weights (A operand: lane (kg, m) holds row m, k = 8 kg .. 8 kg + 7).
  // Layers 1, 2: this wave's output-channel tile tc, segments sA and sA + 2.
  //   layer 1, row tap dy: k = 8 dx + ci (dx < 3), zero for kg = 3;
  //   layer 2, tap 3 dy + dx: k = ci;
  //   layer 3, column tap dx: row m = 4c + dy (c, dy < 3), k = ci.
  const int tc = wv & 1, sA = wv >> 1;
  bf16x8 bw1[3], bw2[9], bw3[3];
#pragma unroll
  for (int dy = 0; dy < 3; dy++)
    bw1[dy] = kg < 3 ? *reinterpret_cast<const bf16x8 *>(w1 + (long)(tc * 16 + m) * KP1 + dy * 24 + kg * 8) : bf16x8{};
#pragma unroll
  for (int tp = 0; tp < 9; tp++)
    bw2[tp] = *reinterpret_cast<const bf16x8 *>(w2 + (long)(tc * 16 + m) * KP2 + tp * 32 + kg * 8);
  const int c3 = m >> 2, dy3 = m & 3;
#pragma unroll
  for (int dx = 0; dx < 3; dx++)
    bw3[dx] = (c3 < C_OUT && dy3 < 3) ? *reinterpret_cast<const bf16x8 *>(w3 + (long)c3 * KP3 + (dy3 * 3 + dx) * 32 + kg * 8)
                                      : bf16x8{};
  f32x4 bv1, bv2;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    bv1[i] = b1[tc * 16 + 4 * kg + i];
    bv2[i] = b2[tc * 16 + 4 * kg + i];
  }
  const float bv3 = kg < C_OUT ? b3[kg] : 0.f;

  const int nsteps = (y1 - y0) + FUSED_HALO;
  // 8-byte part threadIdx.x of input row ri: pixel threadIdx.x / 2 (window
  // column threadIdx.x / 2 - 1), channels 4 (threadIdx.x & 1) .. + 3.  Every
  // lane loads from a clamped address, and what lies outside the image is
  // zeroed when the row is stored to LDS, so each step issues exactly one load
  // per wave and waits only for the load of two steps earlier.
  const int ipx = min((int)threadIdx.x, FIN_PARTS - 1) >> 1, icol = c0 - 1 + ipx;
  const bool iload = icol >= 0 && icol < W;
  const long ioff = ibase * C_INP + (long)min(max(icol, 0), W - 1) * C_INP + 4 * (threadIdx.x & 1);
  auto load_in = [&](int ri) {
    return *reinterpret_cast<const uint2 *>(X + ioff + (long)min(max(ri, 0), H - 1) * W * C_INP);
  };
  const f32x4 zero = {0, 0, 0, 0};
  uint2 in_q[2] = {load_in(y0 - 3), load_in(y0 - 2)};  // rows of steps t, t+1 (slot t % 2)
  f32x4 q3 = zero;  // layer 3 running sums: register dy of lane (c, pixel)
  __syncthreads();

  // KEEP: this wave's 4 channels of the block's own pixels
  auto keep_row = [&](bf16 *__restrict__ dst, int r, int w, uint2 v) {
    if (r >= y0 && r < y1 && w >= 3 && w < FW - 3 && c0 + w < W)
      *reinterpret_cast<uint2 *>(dst + (ibase + (long)r * W + c0 + w) * C_H + tc * 16 + 4 * kg) = v;
  };

  // Step t with ring slot P = t % 2: X completes its rows, Y is one row
  // behind, Z starts.
  auto step = [&](auto SEGS, int t, auto P, FusedRows &Xr, FusedRows &Yr, FusedRows &Zr) {
    constexpr int nu = decltype(SEGS)::value, ws = decltype(P)::value, rs = ws ^ 1;
    // input row y0 - 3 + t -> slot ws, and the load of the row of step t + 2
    if (threadIdx.x < FIN_PARTS) {
      const int ri = y0 - 3 + t;
      const bool in = iload && ri >= 0 && ri < H;
      *reinterpret_cast<uint2 *>(s_in[ws] + 4 * threadIdx.x) = uint2{in ? in_q[ws].x : 0u, in ? in_q[ws].y : 0u};
    }
    in_q[ws] = load_in(y0 - 1 + t);
    // layer 1: input rows y0-3 .. y1+2 (steps 1 .. rows+6); completes row y0-5+t
    // (KEEP runs every layer in every step: what the others skip only reaches
    // rows that nothing reads, and without the branches the kernel keeps to 168
    // registers, three waves per SIMD, not two; a training step 381 -> 365 us
    // with fused_back_kernel likewise.  Plain inference has them either way,
    // and the products skipped are worth more: 55 and 60 us)
    if (KEEP || (t >= 1 && t <= nsteps - 3)) {
      const int r = y0 - 5 + t;
      const bool rin = r >= 0 && r < H;
#pragma unroll
      for (int u = 0; u < nu; u++) {
        const int sg = sA + 2 * u;
        // lanes kg = 3 meet zero weights: they re-read column tap 2
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(s_in[rs] + (16 * sg + m + min(kg, 2)) * C_INP);
        Zr.l1[u] = mfma32(bw1[0], a, bv1);  // a new row's sum starts at its bias
        Yr.l1[u] = mfma32(bw1[1], a, Yr.l1[u]);
        Xr.l1[u] = mfma32(bw1[2], a, Xr.l1[u]);
        const int col = c0 + 16 * sg + m;
        const uint2 v = relu_pack4(Xr.l1[u], rin && col >= 0 && col < W);
        *reinterpret_cast<uint2 *>(s_a1[ws] + (16 * sg + m + 1) * F1S + tc * 16 + 4 * kg) = v;
        if constexpr (KEEP) keep_row(keep1, r, 16 * sg + m, v);
      }
    }
    // layer 2: layer-1 rows y0-2 .. y1+1 (steps 4 .. rows+7); completes row y0-7+t
    if (KEEP || (t >= 4 && t <= nsteps - 2)) {
      const int r = y0 - 7 + t;
      const bool rin = r >= 0 && r < H;
#pragma unroll
      for (int u = 0; u < nu; u++) {
        const int sg = sA + 2 * u;
        bf16x8 a[3];
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
          a[dx] = *reinterpret_cast<const bf16x8 *>(s_a1[rs] + (16 * sg + m + dx) * F1S + kg * 8);
        Zr.l2[u] = mfma32(bw2[0], a[0], bv2);
#pragma unroll
        for (int dx = 1; dx < 3; dx++) Zr.l2[u] = mfma32(bw2[dx], a[dx], Zr.l2[u]);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) Yr.l2[u] = mfma32(bw2[3 + dx], a[dx], Yr.l2[u]);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) Xr.l2[u] = mfma32(bw2[6 + dx], a[dx], Xr.l2[u]);
        const int col = c0 + 16 * sg + m;
        const uint2 v = relu_pack4(Xr.l2[u], rin && col >= 0 && col < W);
        *reinterpret_cast<uint2 *>(s_a2[ws] + (16 * sg + m + 1) * F1S + tc * 16 + 4 * kg) = v;
        if constexpr (KEEP) keep_row(keep2, r, 16 * sg + m, v);
      }
    }
    // layer 3: layer-2 rows y0-1 .. y1 (steps 7 .. rows+8); completes output
    // row y0-9+t, staged from step 9 on
    if ((KEEP || (t >= 7 && t < nsteps)) && (nu == 2 || wv < 2)) {
      const int sg = wv;
      bf16x8 a[3];
#pragma unroll
      for (int dx = 0; dx < 3; dx++)
        a[dx] = *reinterpret_cast<const bf16x8 *>(s_a2[rs] + (16 * sg + m + dx) * F1S + kg * 8);
      f32x4 acc = {0.f, q3[0], q3[1], q3[2]};  // each partial moves on one row tap
#pragma unroll
      for (int dx = 0; dx < 3; dx++) acc = mfma32(bw3[dx], a[dx], acc);
      q3 = acc;
      const int w = 16 * sg + m;
      if (t >= FUSED_HALO && t < nsteps && kg < C_OUT && w >= 3 && w < FW - 3)
        s_out[((t - FUSED_HALO) * FOUT + w - 3) * C_OUT + kg] = acc[2] + bv3;
    }
    // this step's rows become readable, and the slots read in this step may
    // be overwritten in the next
    __syncthreads();
  };

  FusedRows ra, rb, rc;
#pragma unroll
  for (int u = 0; u < 2; u++) ra.l1[u] = rb.l1[u] = rc.l1[u] = ra.l2[u] = rb.l2[u] = rc.l2[u] = zero;
  // whole groups of six steps (the ones past nsteps only load and wait), so
  // every step issues its load and the wait for it is the same on every path
  auto march = [&](auto SEGS) {
    for (int t = 0; t < nsteps; t += 6) {
      step(SEGS, t, IC<0>{}, ra, rb, rc);
      step(SEGS, t + 1, IC<1>{}, rb, rc, ra);
      step(SEGS, t + 2, IC<0>{}, rc, ra, rb);
      step(SEGS, t + 3, IC<1>{}, ra, rb, rc);
      step(SEGS, t + 4, IC<0>{}, rb, rc, ra);
      step(SEGS, t + 5, IC<1>{}, rc, ra, rb);
    }
  };
  // a window whose second half lies outside the image leaves its zeros there
  // (the last of five at 257 columns: a tenth of the products)
  if (c0 + FW / 2 < W) march(IC<2>{});
  else march(IC<1>{});

  // corrected-candidate energy (T != void): this block's U and materials,
  // loaded before the output is written out
  using TE = std::conditional_t<std::is_void_v<T>, float, T>;
  __shared__ double sh[4];
  constexpr int NP = (FUSED_MAX_ROWS * FOUT + 255) / 256;  // points per thread, at most
  const int npt = (y1 - y0) * FOUT;
  TE uv[NP][3], ri[NP], kb[NP];
  const BatchInst<TE> *einst = static_cast<const BatchInst<TE> *>(ea.inst);
  if constexpr (!std::is_void_v<T>) {
    const BatchInst<TE> &d = einst[img];
    // (every load of a thread issued before the first use: the march's
    // registers are free by now, and the loads then wait once, not per point)
#pragma unroll
    for (int n = 0; n < NP; n++) {
      const int p = threadIdx.x + 256 * n;
      const int r = p / FOUT, i = c0 + 3 + (p - r * FOUT), j = y0 + r;
      const long o = p < npt && i < W ? (long)j * d.pitch + d.xoff + i : (long)d.xoff;  // a valid point otherwise
#pragma unroll
      for (int c = 0; c < 3; c++) uv[n][c] = d.U[c * d.plane + o];
      ri[n] = d.rinv ? d.rinv[o] : T(1);
      kb[n] = d.bulk ? d.bulk[o] : T(1);
    }
  }

  // the staged output rows y0 .. y1-1, window columns 3 .. 60
  const int nval = (y1 - y0) * FOUT * C_OUT;
  for (int q = threadIdx.x; q < nval; q += 256) {
    const int r = q / (FOUT * C_OUT), e = q - r * (FOUT * C_OUT);
    const int col = c0 + 3 + e / C_OUT;
    if (col < W) out[(ibase + (long)(y0 + r) * W + c0 + 3) * C_OUT + e] = s_out[q];
  }
  if constexpr (!std::is_void_v<T>) {
    // H-weighted energy of the candidate U + (T)(out_scale * net) at this
    // block's output points (the points outside the corrected region keep U),
    // from the staged values the loop above stored
    const BatchInst<TE> &d = einst[img];
    const double hx = 1.0 / (double)d.hix, hy = 1.0 / (double)d.hiy;
    double acc = 0;
#pragma unroll
    for (int n = 0; n < NP; n++) {
      const int p = threadIdx.x + 256 * n;
      const int r = p / FOUT, i = c0 + 3 + (p - r * FOUT), j = y0 + r;
      if (p >= npt || i >= W) continue;
      const double w = hweight(ea.order, W, i, hx) * hweight(ea.order, H, j, hy);
      const bool on = corrected_at(i, j, W, H, ea.band);
      double v[3];
#pragma unroll
      for (int c = 0; c < 3; c++)
        v[c] = on ? (double)(T)(uv[n][c] + (T)(s_out[p * C_OUT + c] * ea.out_scale[c])) : (double)uv[n][c];
      const double rho = d.rinv ? 1.0 / (double)ri[n] : 1.0;
      const double kinv = d.bulk ? 1.0 / (double)kb[n] : 1.0;
      acc += w * (rho * (v[0] * v[0] + v[1] * v[1]) + kinv * v[2] * v[2]);
    }
    const double sm = block_sum_256(acc, sh);
    if (threadIdx.x == 0) ea.partial[blockIdx.x] = sm;
  }
}

// --------------------------------------------------------------------------
// Fused backward-data: the ReLU-masked gradients of layers 2 and 1,
//   dP2 = [A2 > 0] (W3^T * dY3),   dP1 = [A1 > 0] (W2^T * dP2)
// (* a 3x3 convolution with the mirrored, channel-transposed weights), of one
// image window in one kernel: the march of fused_net_kernel with two layers.
// Both are stored (the weight gradients read them), each block its own rows
// and 58 columns; dP2 also stays in LDS for the second convolution.  The masks
// are fetched two steps ahead like the input row.
//
// Bound: its 290 MB of mask loads and stores and the row march's latency: 80
// us for 16 images of 257^2 (3.6 TB/s).  One convolution launch per layer, its
// FP32 output and a masking launch took 391 us.
// --------------------------------------------------------------------------
// 4 channels of one pixel: bf16, kept where the activation was positive
// (positive and not NaN: bit patterns 1 .. 0x7f80), zero outside the image
__device__ __forceinline__ uint2 mask_pack4(f32x4 acc, uint2 a, bool in)
{
  const unsigned lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{acc[0], acc[1]}, vbf2));
  const unsigned hi = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{acc[2], acc[3]}, vbf2));
  auto keep = [&](unsigned v, unsigned m) {
    const bool k0 = (m & 0xffffu) - 1u < 0x7f80u, k1 = (m >> 16) - 1u < 0x7f80u;
    return (in && k0 ? v & 0xffffu : 0u) | (in && k1 ? v & 0xffff0000u : 0u);
  };
  return uint2{keep(lo, a.x), keep(hi, a.y)};
}

constexpr int BACK_HALO = 6;  // row steps beyond the chunk's rows

__global__ __launch_bounds__(256, 3) void fused_back_kernel(const bf16 *__restrict__ dY3, int H, int W, int rows,
                                                         const bf16 *__restrict__ w3t, const bf16 *__restrict__ w2t,
                                                         const bf16 *__restrict__ A2, const bf16 *__restrict__ A1,
                                                         bf16 *__restrict__ dP2, bf16 *__restrict__ dP1)
{
  __shared__ __attribute__((aligned(16))) bf16 s_in[2][FPX * C_D3];
  __shared__ __attribute__((aligned(16))) bf16 s_a[2][FPX * F1S];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kg = lane >> 4;
  const int strips = (W + FOUT - 1) / FOUT, chunks = (H + rows - 1) / rows;
  const int b = blockIdx.x;
  const int img = b / (strips * chunks), rem = b - img * strips * chunks;
  const int strip = rem / chunks, chunk = rem - strip * chunks;
  const int c0 = strip * FOUT - 3;
  const int y0 = chunk * rows, y1 = min(y0 + rows, H);
  const long ibase = (long)img * H * W;
  for (int q = threadIdx.x; q < 2 * FPX * F1S; q += 256) (&s_a[0][0])[q] = 0;  // the pad pixels stay zero

  const int tc = wv & 1, sA = wv >> 1;
  bf16x8 bw3[3], bw2[9];
#pragma unroll
  for (int dy = 0; dy < 3; dy++)
    bw3[dy] = kg < 3 ? *reinterpret_cast<const bf16x8 *>(w3t + (long)(tc * 16 + m) * KP1 + dy * 24 + kg * 8) : bf16x8{};
#pragma unroll
  for (int tp = 0; tp < 9; tp++)
    bw2[tp] = *reinterpret_cast<const bf16x8 *>(w2t + (long)(tc * 16 + m) * KP2 + tp * 32 + kg * 8);

  const int nsteps = (y1 - y0) + BACK_HALO;
  const int ipx = min((int)threadIdx.x, FIN_PARTS - 1) >> 1, icol = c0 - 1 + ipx;
  const bool iload = icol >= 0 && icol < W;
  const long ioff = ibase * C_D3 + (long)min(max(icol, 0), W - 1) * C_D3 + 4 * (threadIdx.x & 1);
  auto load_in = [&](int ri) {
    return *reinterpret_cast<const uint2 *>(dY3 + ioff + (long)min(max(ri, 0), H - 1) * W * C_D3);
  };
  // this lane's 4 channels of its two pixels, at image row r (clamped: what
  // lies outside is masked when it is used)
  const int ch = tc * 16 + 4 * kg;
  const int col[2] = {c0 + 16 * sA + m, c0 + 16 * (sA + 2) + m};
  long aoff[2];
#pragma unroll
  for (int u = 0; u < 2; u++) aoff[u] = (ibase + min(max(col[u], 0), W - 1)) * C_H + ch;
  auto load_mask = [&](const bf16 *A, int u, int r) {
    return *reinterpret_cast<const uint2 *>(A + aoff[u] + (long)min(max(r, 0), H - 1) * W * C_H);
  };
  const f32x4 zero = {0, 0, 0, 0};
  uint2 in_q[2] = {load_in(y0 - 2), load_in(y0 - 1)};  // rows of steps t, t + 1
  uint2 m2[2][2], m1[2][2];                            // masks of the rows completed in steps t, t + 1
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int u = 0; u < 2; u++) {
      m2[k][u] = load_mask(A2, u, y0 - 4 + k);
      m1[k][u] = load_mask(A1, u, y0 - 6 + k);
    }
  __syncthreads();

  auto step = [&](auto SEGS, int t, auto P, FusedRows &Xr, FusedRows &Yr, FusedRows &Zr) {
    constexpr int nu = decltype(SEGS)::value, ws = decltype(P)::value, rs = ws ^ 1;
    if (threadIdx.x < FIN_PARTS) {
      const int ri = y0 - 2 + t;
      const bool in = iload && ri >= 0 && ri < H;
      *reinterpret_cast<uint2 *>(s_in[ws] + 4 * threadIdx.x) = uint2{in ? in_q[ws].x : 0u, in ? in_q[ws].y : 0u};
    }
    in_q[ws] = load_in(y0 + t);
    uint2 k2[2], k1[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      k2[u] = m2[ws][u];
      k1[u] = m1[ws][u];
      m2[ws][u] = load_mask(A2, u, y0 - 2 + t);
      m1[ws][u] = load_mask(A1, u, y0 - 4 + t);
    }
    // layer 3's transpose: dY3 rows y0-2 .. y1+1 (steps 1 .. rows+4); completes dP2 row y0-4+t
    {
      const int r = y0 - 4 + t;
#pragma unroll
      for (int u = 0; u < nu; u++) {
        const int w = 16 * (sA + 2 * u) + m;
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(s_in[rs] + (w + min(kg, 2)) * C_D3);
        Zr.l1[u] = mfma32(bw3[0], a, zero);
        Yr.l1[u] = mfma32(bw3[1], a, Yr.l1[u]);
        Xr.l1[u] = mfma32(bw3[2], a, Xr.l1[u]);
        const uint2 v = mask_pack4(Xr.l1[u], k2[u], r >= 0 && r < H && col[u] >= 0 && col[u] < W);
        *reinterpret_cast<uint2 *>(s_a[ws] + (w + 1) * F1S + ch) = v;
        if (r >= y0 && r < y1 && w >= 3 && w < FW - 3 && col[u] < W)
          *reinterpret_cast<uint2 *>(dP2 + (ibase + (long)r * W + col[u]) * C_H + ch) = v;
      }
    }
    // layer 2's transpose: dP2 rows y0-1 .. y1 (steps 4 .. rows+5); completes dP1 row y0-6+t
    {
      const int r = y0 - 6 + t;
#pragma unroll
      for (int u = 0; u < nu; u++) {
        const int w = 16 * (sA + 2 * u) + m;
        bf16x8 a[3];
#pragma unroll
        for (int dx = 0; dx < 3; dx++) a[dx] = *reinterpret_cast<const bf16x8 *>(s_a[rs] + (w + dx) * F1S + kg * 8);
        Zr.l2[u] = zero;
#pragma unroll
        for (int dx = 0; dx < 3; dx++) Zr.l2[u] = mfma32(bw2[dx], a[dx], Zr.l2[u]);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) Yr.l2[u] = mfma32(bw2[3 + dx], a[dx], Yr.l2[u]);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) Xr.l2[u] = mfma32(bw2[6 + dx], a[dx], Xr.l2[u]);
        if (r >= y0 && r < y1 && w >= 3 && w < FW - 3 && col[u] < W)
          *reinterpret_cast<uint2 *>(dP1 + (ibase + (long)r * W + col[u]) * C_H + ch) = mask_pack4(Xr.l2[u], k1[u], true);
      }
    }
    __syncthreads();
  };
  FusedRows ra, rb, rc;
#pragma unroll
  for (int u = 0; u < 2; u++) ra.l1[u] = rb.l1[u] = rc.l1[u] = ra.l2[u] = rb.l2[u] = rc.l2[u] = zero;
  auto march = [&](auto SEGS) {
    for (int t = 0; t < nsteps; t += 6) {
      step(SEGS, t, IC<0>{}, ra, rb, rc);
      step(SEGS, t + 1, IC<1>{}, rb, rc, ra);
      step(SEGS, t + 2, IC<0>{}, rc, ra, rb);
      step(SEGS, t + 3, IC<1>{}, ra, rb, rc);
      step(SEGS, t + 4, IC<0>{}, rb, rc, ra);
      step(SEGS, t + 5, IC<1>{}, rc, ra, rb);
    }
  };
  // a window whose second half lies outside the image leaves its zeros there
  if (c0 + FW / 2 < W) march(IC<2>{});
  else march(IC<1>{});
}

// --------------------------------------------------------------------------
// Weight and bias gradients: dW[co][tap][ci] = sum_p dY[p][co] X[p + tap][ci]
// and db[co] = sum_p dY[p][co], as MFMA GEMMs with M = 16 output channels,
// N = 16 input channels (8-channel inputs: 8 channels of two row taps) and the
// sum over pixels as K, 32 per v_mfma_f32_16x16x32_bf16.
//
// The operands lie channels-last in memory and the MFMA wants 8 consecutive
// pixels of one channel per lane, so rows are transposed on their way into
// LDS ([channel][pixel], pairs of pixels packed into dwords) and read back as
// 16-byte fragments.  The three column taps of a fragment are one aligned
// read, its two neighbouring dwords and five v_alignbit; each row of X is
// transposed once and serves three row taps.  A block takes a strip of at most
// WG_PX columns and marches down a chunk of rows, two rows per barrier (waves
// 0, 1 the first, 2, 3 the second; within a pair each wave takes half of the
// input channels, or of the row taps), the next two rows of both operands
// in flight meanwhile.  Accumulators stay in registers over all of a block's
// chunks; the partials are summed in a fixed order (wgrad_reduce_kernel).
//
// Bound: the LDS reads and transposing writes around each row's barrier.  16
// images of 257^2, layers 3 / 2 / 1: 36 / 46 / 28 us; with 2-byte gathers of both operands from global memory and
// 16-pixel MFMAs 651 / 710 / 278 us, and 1228 us more for each layer's bias
// gradient in a kernel of its own.  The reduction of all partials takes 9 us
// (three launches of one serial sum per entry: 271 us each).
// --------------------------------------------------------------------------
constexpr int WG_PX = 96;       // columns of a strip, at most: three groups of 32
constexpr int WG_XS = 120;      // LDS pixels per channel of X: 8 left of the strip, 16-byte rows at an odd multiple
constexpr int WG_DS = 104;      // the same for dY (no halo)
constexpr int WG_BLOCKS = 512;  // partials at most: two blocks per CU

// floats of one partial: [co][tap][ci] of the real output channels, then the bias
constexpr int wg_len(int cin, int cout) { return cout * 9 * cin + cout; }

// how a block's work is cut: strips of `groups` 32-column groups, chunks of `rows` rows
struct WgradGeom {
  int groups, strips, rows, chunks, items;
};
inline WgradGeom wgrad_geom(int nb, int H, int W)
{
  WgradGeom g;
  const int all = (W + 31) / 32;
  g.strips = (all + WG_PX / 32 - 1) / (WG_PX / 32);
  g.groups = (all + g.strips - 1) / g.strips;
  // about one chunk per block, of an even number of at least 8 rows
  const int want = std::max(1, WG_BLOCKS / std::max(1, nb * g.strips));
  g.rows = std::max(8, ((H + want - 1) / want + 1) / 2 * 2);
  g.chunks = (H + g.rows - 1) / g.rows;
  g.items = nb * g.strips * g.chunks;
  return g;
}

// CIN: channels of X (8 or 32); CD: channels of dY in memory (8 or 32), the
// first COUT of them real
template <int CIN, int CD, int COUT>
__global__ __launch_bounds__(256) void wgrad_kernel(const bf16 *__restrict__ X, const bf16 *__restrict__ dY, int H,
                                                    int W, WgradGeom g, float *__restrict__ partial)
{
  static_assert(CIN == 8 || CIN == 32, "input channel tiling");
  constexpr int MT = CD == 32 ? 2 : 1;
  constexpr int NB = CIN == 32 ? 3 : 1;  // B row sets per wave: the three row taps, or one (pair of) row tap(s)
  constexpr int NP = WG_PX / 2 + 2;      // pixel pairs of an X row: columns -2 .. WG_PX + 1
  constexpr int XT = 2 * NP * (CIN / 8), XI = (XT + 255) / 256;          // transposing tasks of two X rows
  constexpr int DT = 2 * (WG_PX / 2) * (CD / 8), DI = (DT + 255) / 256;  // and of two dY rows
  constexpr int XROW = CIN * WG_XS, DROW = CD * WG_DS;
  __shared__ __attribute__((aligned(16))) bf16 smem[6 * XROW + 4 * DROW];
  bf16 *sx = smem, *sd = smem + 6 * XROW;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kg = lane >> 4;
  const int part = wv & 1, half = wv >> 1;

  f32x4 acc[NB][3][MT], bacc[MT];
#pragma unroll
  for (int t = 0; t < MT; t++) {
    bacc[t] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < NB; d++)
#pragma unroll
      for (int x = 0; x < 3; x++) acc[d][x][t] = f32x4{0, 0, 0, 0};
  }
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; i++) ones[i] = (short)0x3f80;  // 1.0

  for (int item = blockIdx.x; item < g.items; item += gridDim.x) {
    const int chunk = item % g.chunks, rest = item / g.chunks;
    const int strip = rest % g.strips, img = rest / g.strips;
    const int x0 = strip * g.groups * 32, wpx = g.groups * 32;
    const int y0 = chunk * g.rows, y1 = min(y0 + g.rows, H);
    const long ibase = (long)img * H * W;

    // two pixels of 8 channels of rows r0 and r0 + 1, zero outside the image
    // (X) or outside this item's pixels (dY)
    auto load_x = [&](int q, int r0, uint4 v[2]) {
      const int r = q / (NP * (CIN / 8)), e = q - r * (NP * (CIN / 8));
      const int row = r0 + r, c = x0 - 2 + 2 * (e / (CIN / 8));
      const bf16 *p = X + (ibase + (long)row * W + c) * CIN + 8 * (e % (CIN / 8));
      const bool in = q < XT && row >= 0 && row < H;
      v[0] = v[1] = uint4{0, 0, 0, 0};
      if (in && c >= 0 && c < W) v[0] = *reinterpret_cast<const uint4 *>(p);
      if (in && c + 1 >= 0 && c + 1 < W) v[1] = *reinterpret_cast<const uint4 *>(p + CIN);
    };
    auto load_d = [&](int q, int r0, uint4 v[2]) {
      const int r = q / (WG_PX / 2 * (CD / 8)), e = q - r * (WG_PX / 2 * (CD / 8));
      const int row = r0 + r, k = 2 * (e / (CD / 8)), c = x0 + k;
      const bf16 *p = dY + (ibase + (long)row * W + c) * CD + 8 * (e % (CD / 8));
      const bool in = q < DT && row < y1 && k < wpx;
      v[0] = v[1] = uint4{0, 0, 0, 0};
      if (in && c < W) v[0] = *reinterpret_cast<const uint4 *>(p);
      if (in && c + 1 < W) v[1] = *reinterpret_cast<const uint4 *>(p + CD);
    };
    // dword (pixel, pixel + 1) of each of the 8 channels
    auto store8 = [](bf16 *dst, int stride, const uint4 v[2]) {
      const unsigned a[4] = {v[0].x, v[0].y, v[0].z, v[0].w}, b[4] = {v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        *reinterpret_cast<unsigned *>(dst + (2 * i) * stride) = (a[i] & 0xffffu) | (b[i] << 16);
        *reinterpret_cast<unsigned *>(dst + (2 * i + 1) * stride) = (a[i] >> 16) | (b[i] & 0xffff0000u);
      }
    };
    auto store_x = [&](int q, int pair, const uint4 v[2]) {  // slots 2 pair, 2 pair + 1
      if (q >= XT) return;
      const int r = q / (NP * (CIN / 8)), e = q - r * (NP * (CIN / 8));
      store8(sx + (2 * pair + r) * XROW + 8 * (e % (CIN / 8)) * WG_XS + 6 + 2 * (e / (CIN / 8)), WG_XS, v);
    };
    auto store_d = [&](int q, int pair, const uint4 v[2]) {
      if (q >= DT) return;
      const int r = q / (WG_PX / 2 * (CD / 8)), e = q - r * (WG_PX / 2 * (CD / 8));
      store8(sd + (2 * pair + r) * DROW + 8 * (e % (CD / 8)) * WG_DS + 2 * (e / (CD / 8)), WG_DS, v);
    };

    __syncthreads();  // the previous item's rows have been read
#pragma unroll
    for (int pr = 0; pr < 2; pr++)
#pragma unroll
      for (int n = 0; n < XI; n++) {
        uint4 v[2];
        load_x(threadIdx.x + 256 * n, y0 - 1 + 2 * pr, v);
        store_x(threadIdx.x + 256 * n, pr, v);
      }
#pragma unroll
    for (int n = 0; n < DI; n++) {
      uint4 v[2];
      load_d(threadIdx.x + 256 * n, y0, v);
      store_d(threadIdx.x + 256 * n, 0, v);
    }
    __syncthreads();

    // rows y, y + 1 of dY against rows y - 1 .. y + 2 of X: X row pairs xs, xs + 1 (mod 3)
    int xs = 0, ds = 0;
    for (int y = y0; y < y1; y += 2) {
      const bool more = y + 2 < y1;
      uint4 qx[XI][2], qd[DI][2];
      if (more) {
#pragma unroll
        for (int n = 0; n < XI; n++) load_x(threadIdx.x + 256 * n, y + 3, qx[n]);
#pragma unroll
        for (int n = 0; n < DI; n++) load_d(threadIdx.x + 256 * n, y + 2, qd[n]);
      }
      const int pn = xs == 2 ? 0 : xs + 1;  // the second row pair
      const bf16 *dr = sd + (2 * ds + half) * DROW;
      // X rows of this wave: row tap d of output row y + half is row y - 1 + half + d
      const bf16 *xr[NB];
      if constexpr (CIN == 32) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const int k = half + d;
          xr[d] = sx + (2 * (k < 2 ? xs : pn) + (k & 1)) * XROW + (part * 16 + m) * WG_XS + 8 + 8 * kg;
        }
      } else {  // part 0: row taps 0 (lanes m < 8) and 1; part 1: row tap 2 (twice)
        const int k = half + (part ? 2 : m >> 3);
        xr[0] = sx + (2 * (k < 2 ? xs : pn) + (k & 1)) * XROW + (m & 7) * WG_XS + 8 + 8 * kg;
      }
      for (int gr = 0; gr < g.groups; gr++) {
        bf16x8 a[MT];
#pragma unroll
        for (int t = 0; t < MT; t++)
          a[t] = *reinterpret_cast<const bf16x8 *>(dr + (CD == 32 ? t * 16 + m : m & 7) * WG_DS + 32 * gr + 8 * kg);
        if (part == 0) {
#pragma unroll
          for (int t = 0; t < MT; t++) bacc[t] = mfma32(a[t], ones, bacc[t]);
        }
#pragma unroll
        for (int d = 0; d < NB; d++) {
          const bf16 *p = xr[d] + 32 * gr;
          const uint4 c = *reinterpret_cast<const uint4 *>(p);
          const unsigned lo = *reinterpret_cast<const unsigned *>(p - 2);
          const unsigned hi = *reinterpret_cast<const unsigned *>(p + 8);
          const unsigned s1 = __builtin_amdgcn_alignbit(c.y, c.x, 16), s2 = __builtin_amdgcn_alignbit(c.z, c.y, 16),
                         s3 = __builtin_amdgcn_alignbit(c.w, c.z, 16);
          const uint4 b[3] = {{__builtin_amdgcn_alignbit(c.x, lo, 16), s1, s2, s3},
                              c,
                              {s1, s2, s3, __builtin_amdgcn_alignbit(hi, c.w, 16)}};
#pragma unroll
          for (int x = 0; x < 3; x++)
#pragma unroll
            for (int t = 0; t < MT; t++) acc[d][x][t] = mfma32(a[t], __builtin_bit_cast(bf16x8, b[x]), acc[d][x][t]);
        }
      }
      if (more) {
        const int pw = pn == 2 ? 0 : pn + 1;
#pragma unroll
        for (int n = 0; n < XI; n++) store_x(threadIdx.x + 256 * n, pw, qx[n]);
#pragma unroll
        for (int n = 0; n < DI; n++) store_d(threadIdx.x + 256 * n, ds ^ 1, qd[n]);
      }
      __syncthreads();
      xs = pn;
      ds ^= 1;
    }
  }

  // the second row's waves hand their sums to the first's
  constexpr int NA = NB * 3 * MT * 4 + MT * 4;
  static_assert(NA * 64 * 2 * (int)sizeof(float) <= (int)sizeof(smem), "accumulators fit the row buffers");
  float *sf = reinterpret_cast<float *>(smem) + part * NA * 64 + lane;
  __syncthreads();
  if (half) {
    int n = 0;
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sf[64 * n++] = bacc[t][i];
#pragma unroll
        for (int d = 0; d < NB; d++)
#pragma unroll
          for (int x = 0; x < 3; x++) sf[64 * n++] = acc[d][x][t][i];
      }
  }
  __syncthreads();
  if (half) return;
  float *P = partial + (long)blockIdx.x * wg_len(CIN, COUT);
  int n = 0;
#pragma unroll
  for (int t = 0; t < MT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int co = t * 16 + 4 * kg + i;
      const float bs = bacc[t][i] + sf[64 * n++];
      if (part == 0 && m == 0 && co < COUT) P[COUT * 9 * CIN + co] = bs;
#pragma unroll
      for (int d = 0; d < NB; d++)
#pragma unroll
        for (int x = 0; x < 3; x++) {
          const float v = acc[d][x][t][i] + sf[64 * n++];
          const int dy = CIN == 32 ? d : (part ? 2 : m >> 3), ci = CIN == 32 ? part * 16 + m : m & 7;
          if (co < COUT && (CIN == 32 || part == 0 || m < 8)) P[(co * 9 + 3 * dy + x) * CIN + ci] = v;
        }
    }
}

// Sums the three layers' partials in a fixed order into the flat gradient
// ([co][ci][ky][kx] weights and biases), and the loss partials.  A block takes
// 64 consecutive partial entries, its 16 waves every 16th partial each.
struct WgradReduce {
  const float *part[3];
  float *gw[3], *gb[3];
  int nparts[3], cin[3], cout[3], first[4];  // first: first block of each layer
  const double *lpart;
  int nl;
  double lscale;
  double *loss;
};

__global__ __launch_bounds__(1024) void wgrad_reduce_kernel(WgradReduce r)
{
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if ((int)blockIdx.x == r.first[3]) {  // the loss: 1024 partials at most, one per thread
    __shared__ double sl[16];
    double s = (int)threadIdx.x < r.nl ? r.lpart[threadIdx.x] : 0.0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) sl[wv] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0;
      for (int k = 0; k < 16; k++) t += sl[k];
      r.loss[0] = t * r.lscale;
    }
    return;
  }
  __shared__ float sh[16][64];
  const int l = (int)blockIdx.x >= r.first[2] ? 2 : ((int)blockIdx.x >= r.first[1] ? 1 : 0);
  const int cin = r.cin[l], cout = r.cout[l], len = wg_len(cin, cout);
  const int e = ((int)blockIdx.x - r.first[l]) * 64 + lane;
  float s = 0.f;
  if (e < len) {
    const float *p = r.part[l] + e;
#pragma unroll 4
    for (int k = wv; k < r.nparts[l]; k += 16) s += p[(long)k * len];
  }
  sh[wv][lane] = s;
  __syncthreads();
  if (wv || e >= len) return;
  s = sh[0][lane];
#pragma unroll
  for (int k = 1; k < 16; k++) s += sh[k][lane];
  const int nw = cout * 9 * cin;
  if (e >= nw) {
    r.gb[l][e - nw] = s;
  } else {
    const int co = e / (9 * cin), rem = e - co * 9 * cin, tap = rem / cin, ci = rem - tap * cin;
    r.gw[l][(co * cin + ci) * 9 + tap] = s;
  }
}

// Gather dataset samples (raw inputs and targets) into a contiguous batch.
__global__ __launch_bounds__(256) void gather_kernel(const float *__restrict__ raw_all, const float *__restrict__ tgt_all,
                                                     const int *__restrict__ idx, int nb, long npix_img,
                                                     const float *__restrict__ shift_scale, const float *__restrict__ out_scale,
                                                     bf16 *__restrict__ X, float *__restrict__ T)
{
  const long p = blockIdx.x * 256L + threadIdx.x;
  if (p >= (long)nb * npix_img) return;
  const int b = (int)(p / npix_img);
  const long q = (long)idx[b] * npix_img + (p - (long)b * npix_img);
#pragma unroll
  for (int c = 0; c < C_INP; c++)
    X[p * C_INP + c] = c < C_IN ? f2bf((raw_all[q * C_IN + c] - shift_scale[c]) * shift_scale[C_IN + c]) : (bf16)0;
#pragma unroll
  for (int c = 0; c < C_OUT; c++) T[p * C_OUT + c] = tgt_all[q * C_OUT + c] / out_scale[c];
}

// Network inputs at grid point (i, j) of a planar acoustic state (u, v, p),
// evaluated in double with every index clamped into the grid:
//   0  rho^-1 * Dx(d4x p)          Dx f = (f[i+1] - f[i-1]) / 2,
//   1  rho^-1 * Dy(d4y p)          d4x f = f[i-2] - 4f[i-1] + 6f[i] - 4f[i+1] + f[i+2]
//   2  K * (Dx(d4x u) + Dy(d4y v))
//   3..5  d4x + d4y of u, v, p
//   6, 7  rho, K
// Channels 0..2 are, up to a constant factor, the leading truncation error
// h^4/30 * d^5/dx^5 of the fourth-order central stencil in each equation of
// the coarse step, so the per-step residual the network predicts is close to
// a linear function of its inputs; 3..7 carry what the next terms and the
// boundary closures need.  All of them are high-pass quantities: the residual
// (about 1e-6 of the state) is far below bf16's resolution of the state.
// The host restatement is corrector.raw_features.
//
// A block packs a PTW x pth<T> tile of one image (taller for FP32 states,
// whose staging takes half the LDS).  The three state planes of the tile
// plus a 3-point halo are staged in LDS (in the state's precision) as
// f[clamp(j)][clamp(i)], so a neighbour read with its index clamped is a
// plain LDS read; the centres of the differenced fourth differences are
// clamped into the image first.  Lane L of a wave owns image column
// x0 - 1 + L and pth/4 consecutive rows: the y-differences of its rows come
// from one window down its column (each fourth difference computed once, not
// once per point that uses it), and the x-differences of the columns beside
// it from the neighbouring lanes by shuffles.  Lanes 0 and 63 are the halo
// columns; lanes 1..62 own the PTW = 62 output columns.
constexpr int PTW = 62, PTX = PTW + 6;
template <typename T> constexpr int pth = sizeof(T) == 4 ? 32 : 16;
template <typename T> constexpr int pty = pth<T> + 6;

// the fourth difference a - 4b + 6c - 4d + e, left to right in double
__device__ __forceinline__ double d4(double a, double b, double c, double d, double e)
{
  return a - 4 * b + 6 * c - 4 * d + e;
}

template <typename T>
__device__ __forceinline__ void pack_tile(const T *__restrict__ U, const T *__restrict__ rinv, const T *__restrict__ bulk,
                                          int nx, int ny, int pitch, int xoff, long plane, int tx, int ty,
                                          const float *__restrict__ shift_scale, bf16 *__restrict__ X,
                                          T (*s)[pty<T>][PTX])
{
  constexpr int PTH = pth<T>, PTY = pty<T>;
  constexpr int RPT = PTH / 4;  // rows per lane
  constexpr int NSTAGE = 3 * PTY * PTX, NLOAD = (NSTAGE + 255) / 256;
  static_assert(PTX == 64 + 4, "one wave of columns plus the stencil's reach");
  const int x0 = tx * PTW, y0 = ty * PTH;
  // every load of the staging is issued before the first LDS store, so the
  // block waits for one memory latency instead of NLOAD of them
  T v[NLOAD];
#pragma unroll
  for (int k = 0; k < NLOAD; k++) {
    const int q = threadIdx.x + 256 * k;
    if (q < NSTAGE) {
      const int c = q / (PTY * PTX), r = q - c * (PTY * PTX);
      const int yy = r / PTX, xx = r - yy * PTX;
      const int gi = min(max(x0 - 3 + xx, 0), nx - 1), gj = min(max(y0 - 3 + yy, 0), ny - 1);
      v[k] = U[c * plane + (long)gj * pitch + xoff + gi];
    }
  }
  const int lane = threadIdx.x & 63;
  const int cx = x0 - 1 + lane;                 // this lane's image column
  const int jb = y0 + (threadIdx.x >> 6) * RPT;  // its first row
  // the material values of this lane's points, loaded with the staging
  T mri[RPT], mK[RPT];
#pragma unroll
  for (int r = 0; r < RPT; r++) {
    const int i = min(max(cx, 0), nx - 1), j = min(jb + r, ny - 1);
    const long o = (long)j * pitch + xoff + i;
    mri[r] = rinv ? rinv[o] : T(1);
    mK[r] = bulk ? bulk[o] : T(1);
  }
#pragma unroll
  for (int k = 0; k < NLOAD; k++) {
    const int q = threadIdx.x + 256 * k;
    if (q < NSTAGE) (&s[0][0][0])[q] = v[k];
  }
  __syncthreads();
  // LDS slot of image column i is i - x0 + 3, of image row j is j - y0 + 3
  auto at = [&](int c, int yy, int xx) { return (double)s[c][yy][xx]; };
  const int xs = lane + 2;                           // this lane's column
  const int xc = min(max(cx, 0), nx - 1) - x0 + 3;  // its centre for x-differences, clamped into the image
  const int yb = jb - y0 + 3;                        // row jb
  // y-differences down the column: p and v at centres jb-1 .. jb+RPT, u at jb .. jb+RPT-1
  double dyp[RPT + 2], dyv[RPT + 2], dyu[RPT];
  {
    double cp[RPT + 6], cv[RPT + 6];
#pragma unroll
    for (int m = 0; m < RPT + 6; m++) {
      cp[m] = at(2, yb - 3 + m, xs);
      cv[m] = at(1, yb - 3 + m, xs);
    }
#pragma unroll
    for (int m = 0; m < RPT + 2; m++) {
      dyp[m] = d4(cp[m], cp[m + 1], cp[m + 2], cp[m + 3], cp[m + 4]);
      dyv[m] = d4(cv[m], cv[m + 1], cv[m + 2], cv[m + 3], cv[m + 4]);
    }
  }
  {
    double cu[RPT + 4];
#pragma unroll
    for (int m = 0; m < RPT + 4; m++) cu[m] = at(0, yb - 2 + m, xs);
#pragma unroll
    for (int m = 0; m < RPT; m++) dyu[m] = d4(cu[m], cu[m + 1], cu[m + 2], cu[m + 3], cu[m + 4]);
  }
  // a centre outside the image takes the nearest image row's value
  if (jb == 0) {
    dyp[0] = dyp[1];
    dyv[0] = dyv[1];
  }
#pragma unroll
  for (int m = 1; m < RPT + 2; m++)
    if (jb - 1 + m > ny - 1) {
      dyp[m] = dyp[m - 1];
      dyv[m] = dyv[m - 1];
    }
  const bool out_lane = lane >= 1 && lane <= PTW && cx < nx;
#pragma unroll
  for (int r = 0; r < RPT; r++) {
    const int yy = yb + r;
    const double dxu = d4(at(0, yy, xc - 2), at(0, yy, xc - 1), at(0, yy, xc), at(0, yy, xc + 1), at(0, yy, xc + 2));
    const double dxv = d4(at(1, yy, xc - 2), at(1, yy, xc - 1), at(1, yy, xc), at(1, yy, xc + 1), at(1, yy, xc + 2));
    const double dxp = d4(at(2, yy, xc - 2), at(2, yy, xc - 1), at(2, yy, xc), at(2, yy, xc + 1), at(2, yy, xc + 2));
    // the x-differences at columns i - 1 and i + 1 (every lane takes part)
    const double dxu_l = __shfl_up(dxu, 1), dxu_r = __shfl_down(dxu, 1);
    const double dxp_l = __shfl_up(dxp, 1), dxp_r = __shfl_down(dxp, 1);
    const int j = jb + r;
    if (!out_lane || j >= ny) continue;
    const int i = cx;
    const double ri = (double)mri[r];
    const double K = (double)mK[r];
    float raw[C_IN];
    raw[0] = (float)(ri * (0.5 * (dxp_r - dxp_l)));
    raw[1] = (float)(ri * (0.5 * (dyp[r + 2] - dyp[r])));
    raw[2] = (float)(K * (0.5 * (dxu_r - dxu_l) + 0.5 * (dyv[r + 2] - dyv[r])));
    raw[3] = (float)(dxu + dyu[r]);
    raw[4] = (float)(dxv + dyv[r + 1]);
    raw[5] = (float)(dxp + dyp[r + 1]);
    raw[6] = (float)(1.0 / ri);
    raw[7] = (float)K;
    __attribute__((aligned(16))) bf16 px[C_INP];
#pragma unroll
    for (int c = 0; c < C_INP; c++) px[c] = f2bf((raw[c] - shift_scale[c]) * shift_scale[C_IN + c]);
    *reinterpret_cast<uint4 *>(X + ((long)j * nx + i) * C_INP) = *reinterpret_cast<const uint4 *>(px);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void pack_state_tiled_kernel(const T *__restrict__ U, const T *__restrict__ rinv,
                                                               const T *__restrict__ bulk, int nx, int ny, int pitch,
                                                               int xoff, long plane,
                                                               const float *__restrict__ shift_scale,
                                                               bf16 *__restrict__ X)
{
  __shared__ T s[3][pty<T>][PTX];  // the state in its own precision (widened exactly)
  const int tiles_x = (nx + PTW - 1) / PTW;
  pack_tile(U, rinv, bulk, nx, ny, pitch, xoff, plane, blockIdx.x % tiles_x, blockIdx.x / tiles_x, shift_scale, X, s);
}

template <typename T>
__global__ __launch_bounds__(256) void pack_batch_tiled_kernel(const BatchInst<T> *__restrict__ inst, int H, int W,
                                                               const float *__restrict__ shift_scale,
                                                               bf16 *__restrict__ X)
{
  __shared__ T s[3][pty<T>][PTX];  // the state in its own precision (widened exactly)
  const int tiles_x = (W + PTW - 1) / PTW, tiles_y = (H + pth<T> - 1) / pth<T>;
  const int k = blockIdx.x / (tiles_x * tiles_y), t = blockIdx.x - k * tiles_x * tiles_y;
  const BatchInst<T> &d = inst[k];
  pack_tile(d.U, d.rinv, d.bulk, W, H, d.pitch, d.xoff, d.plane, t % tiles_x, t / tiles_x, shift_scale,
            X + (long)k * H * W * C_INP, s);
}

// Corrected candidate: Y = U + out_scale * net (into the scratch register).
template <typename T>
__global__ __launch_bounds__(256) void candidate_kernel(const T *__restrict__ U, const float *__restrict__ net, int nx,
                                                        int ny, int pitch, int xoff, long plane, int band,
                                                        const float *__restrict__ out_scale, T *__restrict__ Y)
{
  const long p = blockIdx.x * 256L + threadIdx.x;
  if (p >= (long)nx * ny) return;
  const int j = (int)(p / nx), i = (int)(p - (long)j * nx);
  const long o = (long)j * pitch + xoff + i;
  const bool on = corrected_at(i, j, nx, ny, band);
#pragma unroll
  for (int c = 0; c < 3; c++)
    Y[c * plane + o] = on ? U[c * plane + o] + (T)(net[p * C_OUT + c] * out_scale[c]) : U[c * plane + o];
}

// Accept the candidate when E_new <= E_old * (1 + bound); count rejections.
template <typename T>
__global__ __launch_bounds__(256) void accept_kernel(const T *__restrict__ Y, T *__restrict__ U, long n,
                                                     const double *__restrict__ e_old, const double *__restrict__ e_new,
                                                     double bound, int *__restrict__ rejected)
{
  const bool ok = e_new[0] <= e_old[0] * (1.0 + bound) && e_new[0] == e_new[0];
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i == 0 && !ok) rejected[0] += 1;
  if (ok && i < n) U[i] = Y[i];
}

// ---- batched ensemble (every instance on the corrector's grid) ------------
// Per-instance H-weighted energy of U (which = 0) or of the Y0 scratch
// register (which = 1): blocks [k*bpi, (k+1)*bpi) reduce instance k.
template <typename T>
__global__ __launch_bounds__(256) void batch_energy_kernel(const BatchInst<T> *__restrict__ inst, int bpi, int which,
                                                           int order, double *__restrict__ partial)
{
  __shared__ double sh[4];
  const int k = blockIdx.x / bpi, chunk = blockIdx.x % bpi;
  const BatchInst<T> &d = inst[k];
  const T *u = which ? d.Y0 : d.U;
  const T *comp = which ? nullptr : d.comp;
  const long npts = (long)d.nx * d.ny;
  const double hx = 1.0 / (double)d.hix, hy = 1.0 / (double)d.hiy;
  double acc = 0;
  for (long q = chunk * 256L + threadIdx.x; q < npts; q += (long)bpi * 256) {
    const int j = (int)(q / d.nx), i = (int)(q - (long)j * d.nx);
    const long o = (long)j * d.pitch + d.xoff + i;
    const double w = hweight(order, d.nx, i, hx) * hweight(order, d.ny, j, hy);
    double v[3];
    for (int c = 0; c < 3; c++) {
      double x = (double)u[c * d.plane + o];
      if (comp) x -= (double)comp[c * d.plane + o];
      v[c] = x;
    }
    const double rho = d.rinv ? 1.0 / (double)d.rinv[o] : 1.0;
    const double kinv = d.bulk ? 1.0 / (double)d.bulk[o] : 1.0;
    acc += w * (rho * (v[0] * v[0] + v[1] * v[1]) + kinv * v[2] * v[2]);
  }
  const double s = block_sum_256(acc, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void batch_energy_final_kernel(const double *__restrict__ partial, int count, int bpi, double *__restrict__ e)
{
  const int k = blockIdx.x * 64 + threadIdx.x;
  if (k >= count) return;
  double s = 0;
  for (int b = 0; b < bpi; b++) s += partial[(long)k * bpi + b];
  e[k] = s;
}

// U += (T)(out_scale * net) where the candidate's energy passed the bound
// (the same expression the energy was taken of); count the refusals.  The
// candidate energies are summed here from their per-block partials (bpi per
// instance; each wavefront takes every fourth instance this block touches,
// at most 256 of them).
template <typename T>
__global__ __launch_bounds__(256) void batch_apply_kernel(const BatchInst<T> *__restrict__ inst, int count, int H, int W,
                                                          int band,
                                                          const float *__restrict__ net,
                                                          const float *__restrict__ out_scale,
                                                          const double *__restrict__ e_ref,
                                                          const double *__restrict__ cand_partial, int bpi,
                                                          double bound, int *__restrict__ rejected)
{
  __shared__ bool s_ok[256];
  const long npi = (long)H * W;
  const long p0 = blockIdx.x * 256L;
  const int k0 = (int)(p0 / npi);
  const int k1 = (int)(min(p0 + 255, count * npi - 1) / npi);  // k1 - k0 <= 255
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int k = k0 + wv; k <= k1; k += 4) {
    double e = 0;
    for (int b = lane; b < bpi; b += 64) e += cand_partial[(long)k * bpi + b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
    if (lane == 0) s_ok[k - k0] = e <= e_ref[k] * (1.0 + bound) && e == e;
  }
  __syncthreads();
  const long p = p0 + threadIdx.x;
  if (p >= count * npi) return;
  const int k = (int)(p / npi);
  const long q = p - k * npi;
  const bool ok = s_ok[k - k0];
  if (q == 0 && !ok) rejected[k] += 1;
  const int j = (int)(q / W), i = (int)(q - (long)j * W);
  if (!ok || !corrected_at(i, j, W, H, band)) return;
  const BatchInst<T> &d = inst[k];
  const long o = (long)j * d.pitch + d.xoff + i;
#pragma unroll
  for (int c = 0; c < 3; c++) d.U[c * d.plane + o] = d.U[c * d.plane + o] + (T)(net[p * C_OUT + c] * out_scale[c]);
}

__global__ void clear_ints_kernel(int *__restrict__ p, int n)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void copy_scalar_kernel(const double *__restrict__ s, double *__restrict__ d) { d[0] = s[0]; }

__global__ void clear_int_kernel(int *__restrict__ p) { p[0] = 0; }

int grid_for(long n) { return (int)((n + 255) / 256); }

}  // namespace

struct sbp_corrector {
  int H = 0, W = 0, nb = 0;  // image shape and batch capacity
  int band = 0;              // corrections act on points at least this far from every wall
  hipStream_t stream = nullptr;
  float *params = nullptr, *grads = nullptr, *m = nullptr, *v = nullptr;
  bf16 *w1 = nullptr, *w2 = nullptr, *w3 = nullptr, *w2t = nullptr, *w3t = nullptr;
  float *b1 = nullptr, *b2 = nullptr, *b3 = nullptr;
  float *norm = nullptr;  // NORM_LEN floats: input shift, input scale, output scale
  bf16 *X0 = nullptr, *A1 = nullptr, *A2 = nullptr, *dY3 = nullptr, *dP2 = nullptr, *dP1 = nullptr;
  float *Yo = nullptr, *Tg = nullptr, *wpart = nullptr;
  double *lpart = nullptr, *scalars = nullptr;  // scalars: [0] loss, [1] E_old
  int *rejected = nullptr, *idx = nullptr;
  double *bpart = nullptr, *be_old = nullptr;  // batched energies: per-block partials, reference energies
  double *cpart = nullptr;                      // candidate energies: per-block partials
  int *brej = nullptr;
  float *ds_raw = nullptr, *ds_tgt = nullptr;
  int ds_n = 0;
  long adam_t = 0;
};

namespace {

void release(sbp_corrector *c)
{
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  void *ptrs[] = {c->params, c->grads, c->m, c->v, c->w1, c->w2, c->w3, c->w2t, c->w3t, c->b1, c->b2, c->b3,
                  c->norm, c->X0, c->A1, c->A2, c->dY3, c->dP2, c->dP1, c->Yo, c->Tg, c->wpart,
                  c->lpart, c->scalars, c->rejected, c->idx, c->ds_raw, c->ds_tgt, c->bpart, c->be_old,
                  c->cpart, c->brej};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

template <typename P> int dmalloc(P **p, size_t bytes)
{
  void *q = nullptr;
  if (hipMalloc(&q, std::max<size_t>(bytes, 16)) != hipSuccess) return fail(SBP_ENOMEM, "corrector allocation failed");
  *p = static_cast<P *>(q);
  return SBP_OK;
}

int prepare(sbp_corrector *c)
{
  hipLaunchKernelGGL(prepare_weights_kernel, dim3(grid_for(C_H * KP2)), dim3(256), 0, c->stream, c->params, c->w1,
                     c->w2, c->w3, c->w2t, c->w3t, c->b1, c->b2, c->b3);
  HIP_OR_FAIL(hipGetLastError());
  return SBP_OK;
}

// Network output Yo of the nb packed images X0 (inference: the fused kernel).
// T != void: also the corrected candidate's energy partials (NetEnergyArgs).
template <typename T = void, bool KEEP = false>
void launch_infer(sbp_corrector *c, int nb, hipStream_t stream, NetEnergyArgs ea = NetEnergyArgs{})
{
  const long blocks = (long)nb * net_blocks_per_image(nb, c->H, c->W);
  hipLaunchKernelGGL((fused_net_kernel<T, KEEP>), dim3((unsigned)blocks), dim3(256), 0, stream, c->X0, nb, c->H, c->W,
                     net_chunk_rows(nb, c->H, c->W), c->w1, c->b1, c->w2, c->b2, c->w3, c->b3, c->Yo, c->A1, c->A2, ea);
}

// Training forward of nb images packed in X0: Yo, and the activations A1, A2.
int forward(sbp_corrector *c, int nb)
{
  launch_infer<void, true>(c, nb, c->stream);
  HIP_OR_FAIL(hipGetLastError());
  return SBP_OK;
}

int infer(sbp_corrector *c, int nb)
{
  launch_infer(c, nb, c->stream);
  HIP_OR_FAIL(hipGetLastError());
  return SBP_OK;
}

// One layer's weight and bias gradient partials; returns their number.
template <int CIN, int CD, int COUT> int launch_wgrad(sbp_corrector *c, const bf16 *X, const bf16 *dY, int nb, float *part)
{
  const WgradGeom g = wgrad_geom(nb, c->H, c->W);
  const int blocks = std::min(g.items, WG_BLOCKS);
  hipLaunchKernelGGL((wgrad_kernel<CIN, CD, COUT>), dim3(blocks), dim3(256), 0, c->stream, X, dY, c->H, c->W, g, part);
  return blocks;
}

// Loss against targets Tg and gradients of every parameter into c->grads.
int backward(sbp_corrector *c, int nb)
{
  const long npix = (long)nb * c->H * c->W;
  const int lblocks = (int)std::min<long>(grid_for(npix), 1024);
  const double inv_n = 1.0 / (double)(npix * C_OUT);
  hipLaunchKernelGGL(loss_kernel, dim3(lblocks), dim3(256), 0, c->stream, c->Yo, c->Tg, npix, c->H, c->W, c->band, inv_n,
                     c->dY3, c->lpart);
  hipLaunchKernelGGL(fused_back_kernel, dim3((unsigned)(nb * net_blocks_per_image(nb, c->H, c->W))), dim3(256), 0, c->stream,
                     c->dY3, c->H, c->W, net_chunk_rows(nb, c->H, c->W), c->w3t, c->w2t, c->A2, c->A1, c->dP2, c->dP1);
  WgradReduce r{};
  r.part[0] = c->wpart;
  r.part[1] = r.part[0] + (long)WG_BLOCKS * wg_len(C_INP, C_H);
  r.part[2] = r.part[1] + (long)WG_BLOCKS * wg_len(C_H, C_H);
  r.nparts[2] = launch_wgrad<C_H, C_D3, C_OUT>(c, c->A2, c->dY3, nb, const_cast<float *>(r.part[2]));
  r.nparts[1] = launch_wgrad<C_H, C_H, C_H>(c, c->A1, c->dP2, nb, const_cast<float *>(r.part[1]));
  r.nparts[0] = launch_wgrad<C_INP, C_H, C_H>(c, c->X0, c->dP1, nb, const_cast<float *>(r.part[0]));
  const int cin[3] = {C_INP, C_H, C_H}, cout[3] = {C_H, C_H, C_OUT};
  const int ow[3] = {OFF_W1, OFF_W2, OFF_W3}, ob[3] = {OFF_B1, OFF_B2, OFF_B3};
  for (int l = 0; l < 3; l++) {
    r.cin[l] = cin[l];
    r.cout[l] = cout[l];
    r.gw[l] = c->grads + ow[l];
    r.gb[l] = c->grads + ob[l];
    r.first[l + 1] = r.first[l] + (wg_len(cin[l], cout[l]) + 63) / 64;
  }
  r.lpart = c->lpart;
  r.nl = lblocks;
  r.lscale = inv_n;
  r.loss = c->scalars;
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(r.first[3] + 1), dim3(1024), 0, c->stream, r);
  HIP_OR_FAIL(hipGetLastError());
  return SBP_OK;
}

int check_nb(const sbp_corrector *c, int nb)
{
  if (!c) return fail(SBP_EINVAL, "null corrector");
  if (nb < 1 || nb > c->nb) return fail(SBP_EINVAL, "batch size outside 1..capacity");
  return SBP_OK;
}

}  // namespace

extern "C" {

int sbp_corr_param_count(void) { return N_PARAMS; }

int sbp_corr_create(int nx, int ny, int batch, sbp_corrector **out)
{
  if (!out) return fail(SBP_EINVAL, "null output pointer");
  *out = nullptr;
  if (nx < 3 || ny < 3 || batch < 1 || (long)nx * ny * batch > (1L << 28))
    return fail(SBP_EINVAL, "corrector image or batch size out of range");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(SBP_ENODEV, "no HIP device");
  sbp_corrector *c = new (std::nothrow) sbp_corrector();
  if (!c) return fail(SBP_ENOMEM, "host allocation failed");
  c->H = ny;
  c->W = nx;
  c->nb = batch;
  const long npix = (long)nx * ny * batch;
  int rc = SBP_OK;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) rc = fail(SBP_EHIP, "stream creation failed");
  if (!rc) rc = dmalloc(&c->params, sizeof(float) * N_PARAMS);
  if (!rc) rc = dmalloc(&c->grads, sizeof(float) * N_PARAMS);
  if (!rc) rc = dmalloc(&c->m, sizeof(float) * N_PARAMS);
  if (!rc) rc = dmalloc(&c->v, sizeof(float) * N_PARAMS);
  if (!rc) rc = dmalloc(&c->w1, sizeof(bf16) * C_H * KP1);
  if (!rc) rc = dmalloc(&c->w2, sizeof(bf16) * C_H * KP2);
  if (!rc) rc = dmalloc(&c->w3, sizeof(bf16) * C_OUTP * KP3);
  if (!rc) rc = dmalloc(&c->w2t, sizeof(bf16) * C_H * KP2);
  if (!rc) rc = dmalloc(&c->w3t, sizeof(bf16) * C_H * KP1);
  if (!rc) rc = dmalloc(&c->b1, sizeof(float) * C_H);
  if (!rc) rc = dmalloc(&c->b2, sizeof(float) * C_H);
  if (!rc) rc = dmalloc(&c->b3, sizeof(float) * C_OUTP);
  if (!rc) rc = dmalloc(&c->norm, sizeof(float) * NORM_LEN);
  if (!rc) rc = dmalloc(&c->X0, sizeof(bf16) * npix * C_INP);
  if (!rc) rc = dmalloc(&c->A1, sizeof(bf16) * npix * C_H);
  if (!rc) rc = dmalloc(&c->A2, sizeof(bf16) * npix * C_H);
  if (!rc) rc = dmalloc(&c->dY3, sizeof(bf16) * npix * C_D3);
  if (!rc) rc = dmalloc(&c->dP2, sizeof(bf16) * npix * C_H);
  if (!rc) rc = dmalloc(&c->dP1, sizeof(bf16) * npix * C_H);
  if (!rc) rc = dmalloc(&c->Yo, sizeof(float) * npix * C_OUT);
  if (!rc) rc = dmalloc(&c->Tg, sizeof(float) * npix * C_OUT);
  if (!rc) rc = dmalloc(&c->wpart, sizeof(float) * WG_BLOCKS * (wg_len(C_INP, C_H) + wg_len(C_H, C_H) + wg_len(C_H, C_OUT)));
  if (!rc) rc = dmalloc(&c->lpart, sizeof(double) * 1024);
  if (!rc) rc = dmalloc(&c->scalars, sizeof(double) * 4);
  if (!rc) rc = dmalloc(&c->rejected, sizeof(int));
  if (!rc) rc = dmalloc(&c->idx, sizeof(int) * batch);
  if (!rc) rc = dmalloc(&c->bpart, sizeof(double) * batch * 64);
  if (!rc) rc = dmalloc(&c->cpart, sizeof(double) * batch * net_most_blocks(ny, nx));
  if (!rc) rc = dmalloc(&c->be_old, sizeof(double) * batch);
  if (!rc) rc = dmalloc(&c->brej, sizeof(int) * batch);
  if (!rc) {
    // Default: zero network (identity correction), unit normalisation.
    std::vector<float> zero(N_PARAMS, 0.f);
    std::vector<float> nrm(NORM_LEN, 0.f);
    for (int k = 0; k < C_IN; k++) nrm[C_IN + k] = 1.f;
    for (int k = 0; k < C_OUT; k++) nrm[NORM_OUT + k] = 1.f;
    if (hipMemcpy(c->params, zero.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(c->m, zero.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(c->v, zero.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(c->norm, nrm.data(), sizeof(float) * NORM_LEN, hipMemcpyHostToDevice) != hipSuccess)
      rc = fail(SBP_EHIP, "corrector initialisation failed");
  }
  if (!rc) rc = prepare(c);
  if (!rc && hipStreamSynchronize(c->stream) != hipSuccess) rc = fail(SBP_EHIP, "corrector initialisation failed");
  if (rc) {
    std::string msg = sbp_last_error();
    release(c);
    fail(rc, msg);
    return rc;
  }
  *out = c;
  return SBP_OK;
}

int sbp_corr_destroy(sbp_corrector *c)
{
  release(c);
  return SBP_OK;
}

int sbp_corr_set_params(sbp_corrector *c, const float *params, int n)
{
  if (!c || !params || n != N_PARAMS) return fail(SBP_EINVAL, "parameter vector has the wrong length");
  HIP_OR_FAIL(hipMemcpyAsync(c->params, params, sizeof(float) * N_PARAMS, hipMemcpyHostToDevice, c->stream));
  std::vector<float> zero(N_PARAMS, 0.f);
  HIP_OR_FAIL(hipMemcpyAsync(c->m, zero.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice, c->stream));
  HIP_OR_FAIL(hipMemcpyAsync(c->v, zero.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice, c->stream));
  c->adam_t = 0;
  int rc = prepare(c);
  if (rc) return rc;
  HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  return SBP_OK;
}

int sbp_corr_get_params(sbp_corrector *c, float *params, int n)
{
  if (!c || !params || n != N_PARAMS) return fail(SBP_EINVAL, "parameter vector has the wrong length");
  HIP_OR_FAIL(hipMemcpyAsync(params, c->params, sizeof(float) * N_PARAMS, hipMemcpyDeviceToHost, c->stream));
  HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  return SBP_OK;
}

int sbp_corr_set_normalization(sbp_corrector *c, const float *in_shift, const float *in_scale, const float *out_scale)
{
  if (!c || !in_shift || !in_scale || !out_scale) return fail(SBP_EINVAL, "null argument");
  float nrm[NORM_LEN] = {0};
  for (int k = 0; k < C_IN; k++) {
    nrm[k] = in_shift[k];
    nrm[C_IN + k] = in_scale[k];
  }
  for (int k = 0; k < C_OUT; k++) nrm[NORM_OUT + k] = out_scale[k];
  HIP_OR_FAIL(hipMemcpyAsync(c->norm, nrm, sizeof(nrm), hipMemcpyHostToDevice, c->stream));
  HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  return SBP_OK;
}

// Network output for nb images of raw inputs [nb][ny][nx][C_IN]:
// out [nb][ny][nx][3] in normalised units (multiply by out_scale for the correction).
int sbp_corr_set_band(sbp_corrector *c, int band)
{
  if (!c) return fail(SBP_EINVAL, "null corrector");
  if (band < 0 || 2 * band >= std::min(c->H, c->W)) return fail(SBP_EINVAL, "band leaves no corrected point");
  c->band = band;
  return SBP_OK;
}

int sbp_corr_get_band(const sbp_corrector *c, int *band)
{
  if (!c || !band) return fail(SBP_EINVAL, "null argument");
  *band = c->band;
  return SBP_OK;
}

int sbp_corr_forward(sbp_corrector *c, const float *raw, int nb, float *out)
{
  int rc = check_nb(c, nb);
  if (rc) return rc;
  if (!raw || !out) return fail(SBP_EINVAL, "null argument");
  const long npix = (long)nb * c->H * c->W;
  float *draw = nullptr;
  if ((rc = dmalloc(&draw, sizeof(float) * npix * C_IN))) return rc;
  rc = SBP_OK;
  if (hipMemcpyAsync(draw, raw, sizeof(float) * npix * C_IN, hipMemcpyHostToDevice, c->stream) != hipSuccess)
    rc = fail(SBP_EHIP, "upload failed");
  if (!rc) {
    hipLaunchKernelGGL(pack_raw_kernel, dim3(grid_for(npix)), dim3(256), 0, c->stream, draw, npix, c->norm, c->X0);
    rc = infer(c, nb);
  }
  if (!rc && (hipMemcpyAsync(out, c->Yo, sizeof(float) * npix * C_OUT, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
              hipStreamSynchronize(c->stream) != hipSuccess))
    rc = fail(SBP_EHIP, "forward failed");
  (void)hipFree(draw);
  return rc;
}

// Loss and parameter gradients for nb images (raw inputs, targets in
// physical units [nb][ny][nx][3]); grads has sbp_corr_param_count() entries.
int sbp_corr_gradients(sbp_corrector *c, const float *raw, const float *target, int nb, float *grads, double *loss)
{
  int rc = check_nb(c, nb);
  if (rc) return rc;
  if (!raw || !target || !grads) return fail(SBP_EINVAL, "null argument");
  const long npix = (long)nb * c->H * c->W;
  float *draw = nullptr, *dtgt = nullptr;
  if ((rc = dmalloc(&draw, sizeof(float) * npix * C_IN))) return rc;
  if ((rc = dmalloc(&dtgt, sizeof(float) * npix * C_OUT))) {
    (void)hipFree(draw);
    return rc;
  }
  std::vector<int> idx(nb);
  for (int b = 0; b < nb; b++) idx[b] = b;
  rc = SBP_OK;
  if (hipMemcpyAsync(draw, raw, sizeof(float) * npix * C_IN, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
      hipMemcpyAsync(dtgt, target, sizeof(float) * npix * C_OUT, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
      hipMemcpyAsync(c->idx, idx.data(), sizeof(int) * nb, hipMemcpyHostToDevice, c->stream) != hipSuccess)
    rc = fail(SBP_EHIP, "upload failed");
  if (!rc) {
    hipLaunchKernelGGL(gather_kernel, dim3(grid_for(npix)), dim3(256), 0, c->stream, draw, dtgt, c->idx, nb,
                       (long)c->H * c->W, c->norm, c->norm + NORM_OUT, c->X0, c->Tg);
    rc = forward(c, nb);
  }
  if (!rc) rc = backward(c, nb);
  double l = 0;
  if (!rc && (hipMemcpyAsync(grads, c->grads, sizeof(float) * N_PARAMS, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
              hipMemcpyAsync(&l, c->scalars, sizeof(double), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
              hipStreamSynchronize(c->stream) != hipSuccess))
    rc = fail(SBP_EHIP, "gradient download failed");
  if (!rc && loss) *loss = l;
  (void)hipFree(draw);
  (void)hipFree(dtgt);
  return rc;
}

// Resident training set: raw inputs [n][ny][nx][5] and targets [n][ny][nx][3].
int sbp_corr_load_dataset(sbp_corrector *c, const float *raw, const float *target, int n)
{
  if (!c || !raw || !target || n < 1) return fail(SBP_EINVAL, "bad dataset");
  HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  if (c->ds_raw) (void)hipFree(c->ds_raw);
  if (c->ds_tgt) (void)hipFree(c->ds_tgt);
  c->ds_raw = nullptr;
  c->ds_tgt = nullptr;
  c->ds_n = 0;
  const long npix = (long)n * c->H * c->W;
  int rc;
  if ((rc = dmalloc(&c->ds_raw, sizeof(float) * npix * C_IN)) || (rc = dmalloc(&c->ds_tgt, sizeof(float) * npix * C_OUT)))
    return rc;
  HIP_OR_FAIL(hipMemcpy(c->ds_raw, raw, sizeof(float) * npix * C_IN, hipMemcpyHostToDevice));
  HIP_OR_FAIL(hipMemcpy(c->ds_tgt, target, sizeof(float) * npix * C_OUT, hipMemcpyHostToDevice));
  c->ds_n = n;
  return SBP_OK;
}

// One Adam step on the mini-batch idx[0..nb) of the resident dataset.
int sbp_corr_train_step(sbp_corrector *c, const int *idx, int nb, float lr, double *loss)
{
  int rc = check_nb(c, nb);
  if (rc) return rc;
  if (!idx || c->ds_n == 0) return fail(SBP_ESTATE, "no dataset loaded");
  for (int b = 0; b < nb; b++)
    if (idx[b] < 0 || idx[b] >= c->ds_n) return fail(SBP_EINVAL, "sample index out of range");
  const long npix = (long)nb * c->H * c->W;
  HIP_OR_FAIL(hipMemcpyAsync(c->idx, idx, sizeof(int) * nb, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(gather_kernel, dim3(grid_for(npix)), dim3(256), 0, c->stream, c->ds_raw, c->ds_tgt, c->idx, nb,
                     (long)c->H * c->W, c->norm, c->norm + NORM_OUT, c->X0, c->Tg);
  if ((rc = forward(c, nb)) || (rc = backward(c, nb))) return rc;
  c->adam_t++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)c->adam_t), c2 = 1.f - std::pow(b2, (float)c->adam_t);
  hipLaunchKernelGGL(adam_kernel, dim3(grid_for(N_PARAMS)), dim3(256), 0, c->stream, c->params, c->m, c->v, c->grads,
                     N_PARAMS, lr, b1, b2, 1e-8f, c1, c2);
  HIP_OR_FAIL(hipGetLastError());
  if ((rc = prepare(c))) return rc;
  if (loss) {
    HIP_OR_FAIL(hipMemcpyAsync(loss, c->scalars, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  }
  return SBP_OK;
}

int sbp_corr_synchronize(sbp_corrector *c)
{
  if (!c) return fail(SBP_EINVAL, "null corrector");
  HIP_OR_FAIL(hipStreamSynchronize(c->stream));
  return SBP_OK;
}

// Correct the resident state of a 2D acoustic context in place after a step:
// U <- U + out_scale * net(features of U, rho, K), unless the corrected
// state's discrete energy exceeds the reference energy (c->scalars[1]) times
// (1 + bound), in which case the plain step is kept.
static int apply_one(sbp_corrector *c, sbp_ctx *x, double bound)
{
  const long npix = (long)x->nx * x->ny;
  const float *ss = c->norm;
  const int pth_ = x->esz == 8 ? pth<double> : pth<float>;
  const unsigned ptiles = (unsigned)(((x->nx + PTW - 1) / PTW) * ((x->ny + pth_ - 1) / pth_));
  if (x->esz == 8)
    hipLaunchKernelGGL(pack_state_tiled_kernel<double>, dim3(ptiles), dim3(256), 0, x->stream, (const double *)x->U,
                       (const double *)x->rinv, (const double *)x->bulk, x->nx, x->ny, x->pitch, x->xoff, x->plane, ss,
                       c->X0);
  else
    hipLaunchKernelGGL(pack_state_tiled_kernel<float>, dim3(ptiles), dim3(256), 0, x->stream, (const float *)x->U,
                       (const float *)x->rinv, (const float *)x->bulk, x->nx, x->ny, x->pitch, x->xoff, x->plane, ss,
                       c->X0);
  HIP_OR_FAIL(hipGetLastError());
  // the network runs on the context's stream so steps and corrections stay ordered
  hipStream_t keep = c->stream;
  c->stream = x->stream;
  int rc = infer(c, 1);
  c->stream = keep;
  if (rc) return rc;
  // candidate into the Y0 scratch register; its energy lands in x->scalar and
  // is compared with the reference energy (c->scalars[1])
  if (x->esz == 8)
    hipLaunchKernelGGL(candidate_kernel<double>, dim3(grid_for(npix)), dim3(256), 0, x->stream, (const double *)x->U,
                       c->Yo, x->nx, x->ny, x->pitch, x->xoff, x->plane, c->band, c->norm + NORM_OUT, (double *)x->Y0);
  else
    hipLaunchKernelGGL(candidate_kernel<float>, dim3(grid_for(npix)), dim3(256), 0, x->stream, (const float *)x->U,
                       c->Yo, x->nx, x->ny, x->pitch, x->xoff, x->plane, c->band, c->norm + NORM_OUT, (float *)x->Y0);
  HIP_OR_FAIL(hipGetLastError());
  if ((rc = sbp::host::energy_of(x, x->Y0, x->KC, nullptr))) return rc;
  const long n = 3 * x->plane;
  if (x->esz == 8)
    hipLaunchKernelGGL(accept_kernel<double>, dim3(grid_for(n)), dim3(256), 0, x->stream, (const double *)x->Y0,
                       (double *)x->U, n, c->scalars + 1, x->scalar, bound, c->rejected);
  else
    hipLaunchKernelGGL(accept_kernel<float>, dim3(grid_for(n)), dim3(256), 0, x->stream, (const float *)x->Y0,
                       (float *)x->U, n, c->scalars + 1, x->scalar, bound, c->rejected);
  HIP_OR_FAIL(hipGetLastError());
  return SBP_OK;
}

// nsteps coarse RK4 steps of ctx, each followed by the guarded correction.
// The reference energy is the state's energy when the call starts: with
// energy-stable boundary conditions and no forcing the exact solution keeps
// it, so a correction that lifts the energy above it by more than the
// relative bound is growth the scheme cannot have, and is refused.
// *rejected receives the number of corrections refused by the energy bound.
int sbp_corr_advance(sbp_corrector *c, sbp_ctx *x, double t0, double dt, long nsteps, double bound, int *rejected)
{
  if (!c || !x) return fail(SBP_EINVAL, "null argument");
  if (x->phys != SBP_ACOUSTIC_2D) return fail(SBP_EINVAL, "the corrector acts on 2D acoustic contexts");
  if (x->prec == SBP_FP32_KAHAN) return fail(SBP_EINVAL, "the corrector acts on FP64 or FP32 contexts");
  if (x->nx != c->W || x->ny != c->H) return fail(SBP_EINVAL, "context grid differs from the corrector's");
  if (!x->have_state) return fail(SBP_ESTATE, "no state loaded");
  if (!(bound >= 0)) return fail(SBP_EINVAL, "energy bound must be >= 0");
  hipLaunchKernelGGL(clear_int_kernel, dim3(1), dim3(1), 0, x->stream, c->rejected);
  // reference energy: the state's energy when the call starts -> c->scalars[1]
  int rc = sbp::host::energy_of(x, x->U, x->KC, nullptr);
  if (rc) return rc;
  hipLaunchKernelGGL(copy_scalar_kernel, dim3(1), dim3(1), 0, x->stream, x->scalar, c->scalars + 1);
  double t = t0;
  for (long s = 0; s < nsteps; s++) {
    HIP_OR_FAIL(sbp::host::launch_step(x, t, dt));
    rc = apply_one(c, x, bound);
    if (rc) return rc;
    t = t + dt;
  }
  int rej = 0;
  HIP_OR_FAIL(hipMemcpyAsync(&rej, c->rejected, sizeof(int), hipMemcpyDeviceToHost, x->stream));
  HIP_OR_FAIL(hipStreamSynchronize(x->stream));
  if (rejected) *rejected = rej;
  return SBP_OK;
}

// nsteps RK4 steps of every instance of a batch, each followed by the
// guarded correction of every instance (one network pass over all of them).
// Every instance must have the corrector's grid; rejected[k] (count entries,
// optional) receives the corrections refused for instance k.
int sbp_corr_advance_batch(sbp_corrector *c, sbp_batch *b, const double *dt, long nsteps, double bound,
                           int *rejected)
{
  if (!c || !b || !dt) return fail(SBP_EINVAL, "null argument");
  if (b->count > c->nb) return fail(SBP_EINVAL, "batch larger than the corrector's capacity");
  if (b->prec == SBP_FP32_KAHAN) return fail(SBP_EINVAL, "the corrector acts on FP64 or FP32 batches");
  for (int k = 0; k < b->count; k++) {
    if (b->inst[k].nx != c->W || b->inst[k].ny != c->H)
      return fail(SBP_EINVAL, "every instance must have the corrector's grid");
    if (!b->have_state[k]) return fail(SBP_ESTATE, "every instance needs a state");
  }
  if (!(bound >= 0)) return fail(SBP_EINVAL, "energy bound must be >= 0");
  int rc = sbp::host::batch_upload_dt(b, dt);
  if (rc) return rc;
  const int count = b->count, bpi = 64;
  // candidate-energy partials per instance: one per inference block
  const int cbpi = (int)net_blocks_per_image(count, c->H, c->W);
  const int pth_ = b->esz == 8 ? pth<double> : pth<float>;
  const int ptiles = ((c->W + PTW - 1) / PTW) * ((c->H + pth_ - 1) / pth_);
  const long npix = (long)count * c->H * c->W;
  hipStream_t s = b->stream;
  hipLaunchKernelGGL(clear_ints_kernel, dim3((count + 255) / 256), dim3(256), 0, s, c->brej, count);
  // reference energy of every instance: its energy when the call starts
  if (b->esz == 8)
    hipLaunchKernelGGL(batch_energy_kernel<double>, dim3(count * bpi), dim3(256), 0, s,
                       static_cast<const BatchInst<double> *>(sbp::host::batch_inst(b)), bpi, 0, b->order, c->bpart);
  else
    hipLaunchKernelGGL(batch_energy_kernel<float>, dim3(count * bpi), dim3(256), 0, s,
                       static_cast<const BatchInst<float> *>(sbp::host::batch_inst(b)), bpi, 0, b->order, c->bpart);
  hipLaunchKernelGGL(batch_energy_final_kernel, dim3((count + 63) / 64), dim3(64), 0, s, c->bpart, count, bpi, c->be_old);
  HIP_OR_FAIL(hipGetLastError());
  // one corrected step: plain RK4 stages, features, network, candidate
  // energy, guarded update
  // (descriptors of the parity after the step: a two-stage step moves the
  // state into the Y0 pool)
  auto enqueue_step = [&]() -> hipError_t {
    hipError_t e = sbp::host::batch_launch_step(b);
    if (e != hipSuccess) return e;
    if (b->esz == 8) {
      const BatchInst<double> *inst = static_cast<const BatchInst<double> *>(sbp::host::batch_inst(b));
      hipLaunchKernelGGL(pack_batch_tiled_kernel<double>, dim3(count * ptiles), dim3(256), 0, s, inst, c->H, c->W,
                         c->norm, c->X0);
      launch_infer<double>(c, count, s, NetEnergyArgs{inst, c->norm + NORM_OUT, c->cpart, b->order, c->band});
      hipLaunchKernelGGL(batch_apply_kernel<double>, dim3(grid_for(npix)), dim3(256), 0, s, inst, count, c->H, c->W,
                         c->band, c->Yo, c->norm + NORM_OUT, c->be_old, c->cpart, cbpi, bound, c->brej);
    } else {
      const BatchInst<float> *inst = static_cast<const BatchInst<float> *>(sbp::host::batch_inst(b));
      hipLaunchKernelGGL(pack_batch_tiled_kernel<float>, dim3(count * ptiles), dim3(256), 0, s, inst, c->H, c->W,
                         c->norm, c->X0);
      launch_infer<float>(c, count, s, NetEnergyArgs{inst, c->norm + NORM_OUT, c->cpart, b->order, c->band});
      hipLaunchKernelGGL(batch_apply_kernel<float>, dim3(grid_for(npix)), dim3(256), 0, s, inst, count, c->H, c->W,
                         c->band, c->Yo, c->norm + NORM_OUT, c->be_old, c->cpart, cbpi, bound, c->brej);
    }
    return hipGetLastError();
  };
  // (launched one by one: a step's four kernels take longer than their launches
  // even for one small image, and a captured graph of them would be instantiated
  // on every call: 32 steps of one 257^2 image 2080 us launched, 2235 replayed)
  for (long k = 0; k < nsteps; k++) HIP_OR_FAIL(enqueue_step());
  std::vector<int> rej(count, 0);
  HIP_OR_FAIL(hipMemcpyAsync(rej.data(), c->brej, sizeof(int) * count, hipMemcpyDeviceToHost, s));
  HIP_OR_FAIL(hipStreamSynchronize(s));
  if (rejected) std::memcpy(rejected, rej.data(), sizeof(int) * count);
  return SBP_OK;
}

}  // extern "C"
