// akx_surrogate.hip -- training set, training and evaluation of the
// constitutive surrogate (akx_mlp.hpp) on gfx950 matrix cores.
//
// The plain law it stands in for is the neo-Hookean energy/stress
// (material_neohookean_inline_impl.hh:46-65, 145-158) under the Marigo damage
// update (material_marigo_inline_impl.hh:67-76).  The damage update itself
// stays closed-form: it needs the point's own threshold Yd, which no network
// input carries, so the network returns the undamaged stress and the driving
// energy Y = W_NH, and the caller applies d_new = min(1, (Y - Yd) / Sd) when
// Y - Yd - Sd d > 0 and S = (1 - d_new) S_NH exactly as the plain law does.
//
// Training: minibatch Adam on the mean squared error of the scaled outputs,
// FP32 master weights, BF16 MFMA for every product of the forward and the
// backward pass (FP32 accumulation), deterministic reductions (fixed-order
// split-K partial sums, no floating-point atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "akx_internal.hpp"
#include "akx_mlp.hpp"

namespace akx {
using namespace mlp;

namespace {

// ---------------------------------------------------------------------------
// counter-based random numbers (SplitMix64 finaliser) for the path generator
// and the minibatch draws
__host__ __device__ inline uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
struct Rng {
  uint64_t s;
  __device__ double uniform() {  // (0, 1)
    s = mix64(s);
    return (double((s >> 11)) + 0.5) * (1.0 / 9007199254740992.0);
  }
  __device__ double normal() {
    const double u1 = uniform(), u2 = uniform();
    return sqrt(-2. * log(u1)) * cos(6.283185307179586 * u2);
  }
};

// Neo-Hookean PK2 stress (Voigt) and energy from the Green-Lagrange strain:
// C = I + 2E, J = sqrt(det C), S = mu (I - C^-1) + lambda ln J C^-1,
// W = lambda/2 ln^2 J + mu (-ln J + (tr C - 3)/2).
__device__ inline void nh_green(const double* E, double lambda, double mu, double* S, double* W) {
  const double c00 = 1 + 2 * E[0], c11 = 1 + 2 * E[1], c22 = 1 + 2 * E[2];
  const double c12 = 2 * E[3], c02 = 2 * E[4], c01 = 2 * E[5];
  const double a00 = c11 * c22 - c12 * c12, a11 = c00 * c22 - c02 * c02,
               a22 = c00 * c11 - c01 * c01;
  const double a12 = c02 * c01 - c00 * c12, a02 = c01 * c12 - c11 * c02,
               a01 = c12 * c02 - c01 * c22;
  const double det = c00 * a00 + c01 * a01 + c02 * a02;
  const double lnJ = 0.5 * log(det);
  const double id = 1. / det;
  const double ci[6] = {a00 * id, a11 * id, a22 * id, a12 * id, a02 * id, a01 * id};
  const double f = lambda * lnJ - mu;
  S[0] = mu + f * ci[0];
  S[1] = mu + f * ci[1];
  S[2] = mu + f * ci[2];
  S[3] = f * ci[3];
  S[4] = f * ci[4];
  S[5] = f * ci[5];
  *W = 0.5 * lambda * lnJ * lnJ + mu * (-lnJ + 0.5 * (c00 + c11 + c22 - 3.));
}

__device__ inline void linear_part(const double* E, double lambda, double mu, double* S,
                                   double* W) {
  const double tr = E[0] + E[1] + E[2];
  for (int k = 0; k < 3; ++k) S[k] = lambda * tr + 2 * mu * E[k];
  for (int k = 3; k < 6; ++k) S[k] = 2 * mu * E[k];
  const double ee = E[0] * E[0] + E[1] * E[1] + E[2] * E[2] +
                    2 * (E[3] * E[3] + E[4] * E[4] + E[5] * E[5]);
  *W = 0.5 * lambda * tr * tr + mu * ee;
}

// ---------------------------------------------------------------------------
// training set: one thread per strain path.  Monotone paths drift along a
// fixed random direction, cyclic paths reverse it every `period` steps; both
// add Gaussian increments and reflect at |E_k| = eps.  The damage follows the
// Marigo update with a per-path Weibull threshold.
__global__ void __launch_bounds__(256) k_sur_gen(int64_t paths, int steps, double eps,
                                                 double inc_std, double lambda, double mu,
                                                 double Sd, double yd_scale, double yd_shape,
                                                 double sS, double sW, uint64_t seed, float* X,
                                                 float* T) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= paths) return;
  Rng r{mix64(seed ^ (uint64_t(p) * 0xD1B54A32D192ED03ull))};
  const bool cyclic = r.uniform() < 0.5;
  double dir[6], nrm = 0;
  for (int k = 0; k < 6; ++k) {
    dir[k] = r.normal();
    nrm += dir[k] * dir[k];
  }
  nrm = sqrt(nrm);
  for (int k = 0; k < 6; ++k) dir[k] /= nrm;
  const double drift = inc_std * (0.5 + 2.5 * r.uniform());
  const int period = 10 + int(40 * r.uniform());
  const double Yd = yd_scale * pow(-log(r.uniform()), 1. / yd_shape);
  double E[6] = {0, 0, 0, 0, 0, 0};
  double d = 0;
  for (int s = 0; s < steps; ++s) {
    const double sg = (cyclic && ((s / period) & 1)) ? -1. : 1.;
    for (int k = 0; k < 6; ++k) {
      double v = E[k] + sg * drift * dir[k] + inc_std * r.normal();
      if (v > eps) v = 2 * eps - v;
      if (v < -eps) v = -2 * eps - v;
      E[k] = fmin(eps, fmax(-eps, v));
    }
    double S[6], W, Sl[6], Wl;
    nh_green(E, lambda, mu, S, &W);
    linear_part(E, lambda, mu, Sl, &Wl);
    const int64_t q = p * steps + s;
    for (int k = 0; k < 6; ++k) X[q * 7 + k] = float(E[k] / eps);
    X[q * 7 + 6] = float(d);
    for (int k = 0; k < 6; ++k) T[q * 7 + k] = float((S[k] - Sl[k]) / sS);
    T[q * 7 + 6] = float((W - Wl) / sW);
    // material_marigo_inline_impl.hh:67-76 with Y = W_NH
    const double Fd = W - Yd - Sd * d;
    if (Fd > 0) d = (W - Yd) / Sd;
    d = fmin(d, 1.);
  }
}

// ---------------------------------------------------------------------------
// Training pass.  Three launches per minibatch: k_sur_pass (draw, forward,
// output error, backward through the layers), k_sur_weight_gradients (every
// layer's split-K products) and k_sur_update.  16-bit operands live in memory
// as MFMA fragments, so that every operand load is one contiguous kilobyte per
// wave:
//   weights, rows x K:      frag(row, k, K / 16), both orientations
//   activations and errors: [16-point group][feature][point], K = points
__host__ __device__ constexpr int frag(int row, int k, int ksteps) {
  return (((row >> 5) * ksteps + (k >> 4)) * 64 + ((k >> 3) & 1) * 32 + (row & 31)) * 8 + (k & 7);
}
// features stored per 16-point group: the inputs (7 + 7 residuals + 2 zeros),
// the hidden layers, and the output errors (7 + 1 zero)
__host__ __device__ constexpr int act_rows(int layer) { return layer == 0 ? K0 : HID; }
__host__ __device__ constexpr int err_rows(int layer) { return layer == 4 ? 8 : HID; }

struct PassArgs {
  const float *X, *T;       // samples: n x 7 inputs and targets
  int64_t n;
  int B;                    // batch (a multiple of 32)
  uint64_t seed;
  int64_t iter;
  int draw;                 // samples drawn with replacement, else sample b
  const __bf16* W[5];       // weights, fragments
  const __bf16* WT[5];      // transposed weights (layers 1 to 4)
  const float* params;      // biases
  __bf16* act[5];           // inputs of layer l (l = 0: the samples), point groups
  __bf16* err[5];           // errors at the output of layer l
  float *Y, *T8;            // outputs and targets, B x 8 (nullptr: not written)
  int backward;
};

// One block of 4 waves per 32 points; wave mb owns features 32 mb .. 32 mb + 31
// of every layer.  A layer's result tile becomes the next layer's operand
// through LDS (rows of 128 + 8: 16-byte reads without bank conflicts); the
// pre-activations stay in registers for the way back, whose tiles have the
// same shape.  Products, roundings and their order are those of one 32 x 32
// tile per wave and layer, so the pass is bound by the chain of its layers
// (LDS exchange, barrier, 8 MFMAs), not by rates: 12 us at a batch of 8,192,
// and 7 more for the 17 MB of activations and errors the weight gradients
// read.  As one launch per layer and direction, with every intermediate
// written twice (row-major and transposed), such a minibatch took 205 us of
// kernels in 21 launches, now 32 in three.  One wave per SIMD with all its
// registers: capped at two (spilling) it was slower at every batch (8,192: 48
// against 35 us per minibatch, 65,536: 222 against 161).
__global__ void __launch_bounds__(256) k_sur_pass(PassArgs A) {
  constexpr int HS = HID + 8, XS = 24, TS = 40;
  __shared__ __align__(16) __bf16 s_h[2][32][HS];
  __shared__ __align__(16) __bf16 s_x[32][XS];      // inputs, later output errors
  __shared__ __align__(16) __bf16 s_t[4][32][TS];   // a wave's tile, transposed
  __shared__ __align__(16) float s_b[4 * HID + 8];
  __shared__ float s_T[32][8];
  const int64_t tile = blockIdx.x;
  const int mb = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5;
  constexpr int OFF_B[5] = {OFF_B0, OFF_B1, OFF_B2, OFF_B3, OFF_B4};
  // the weights of the layer after the current one, loaded a layer ahead
  bf16x8 w[8], wn[8];
  auto fetch = [&](const __bf16* W, int ksteps, bf16x8 (&dst)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (t < ksteps)
        dst[t] = *reinterpret_cast<const bf16x8*>(W + ((mb * ksteps + t) * 64 + lane) * 8);
  };
  fetch(A.W[0], 1, w);
  fetch(A.W[1], 8, wn);
  if (threadIdx.x < 32) {
    const int64_t b = tile * 32 + threadIdx.x;
    const int64_t idx =
        A.draw ? int64_t(mix64(A.seed ^ mix64(uint64_t(A.iter) * A.B + b)) % uint64_t(A.n)) : b;
    float x[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) x[k] = A.X[idx * NIN + k];
#pragma unroll
    for (int k = 0; k < K0; ++k) {
      float v = 0.f;
      if (k < NIN) v = x[k];
      else if (k < 2 * NIN) v = x[k - NIN] - from_bf16(to_bf16(x[k - NIN]));
      const __bf16 bv = to_bf16(v);
      s_x[threadIdx.x][k] = bv;
      if (A.backward)
        A.act[0][((b >> 4) * K0 + k) * 16 + (b & 15)] = bv;
    }
#pragma unroll
    for (int k = 0; k < NOUT; ++k) s_T[threadIdx.x][k] = A.T[idx * NOUT + k];
    s_T[threadIdx.x][7] = 0.f;
  } else {
    for (int k = int(threadIdx.x) - 32; k < 4 * HID + NOUT; k += 224) {
      const int l = k >> 7;
      s_b[k] = A.params[OFF_B[l] + (k - l * HID)];
    }
  }
  lds_barrier();
  // a wave's tile of 16-bit values v[16] (register r: feature 32 mb +
  // crow(r, h), point i): to s_h[buf] for the next layer and, transposed
  // through LDS, to memory for the weight gradients
  auto emit = [&](const __bf16 (&v)[16], int buf, __bf16* out, int rows) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
      *reinterpret_cast<bf16x4*>(&s_h[buf][i][32 * mb + crow(4 * g, h)]) =
          bf16x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
    }
    if (A.backward) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s_t[mb][crow(r, h)][i] = v[r];
    }
    lds_barrier();
    if (A.backward) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int row = lane >> 1, half = lane & 1;
        const bf16x8 u = *reinterpret_cast<const bf16x8*>(&s_t[mb][row][16 * g + 8 * half]);
        *reinterpret_cast<bf16x8*>(out + ((tile * 2 + g) * rows + 32 * mb + row) * 16 + 8 * half) =
            u;
      }
    }
  };
  auto product = [&](const bf16x8 (&a)[8], int buf) {
    f32x16 acc = f32x16{};
#pragma unroll
    for (int t = 0; t < 8; ++t)
      acc = mfma(a[t], *reinterpret_cast<const bf16x8*>(&s_h[buf][i][16 * t + 8 * h]), acc);
    return acc;
  };
  f32x16 z[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    f32x16 acc;
    if (l == 0) acc = mfma(w[0], *reinterpret_cast<const bf16x8*>(&s_x[i][8 * h]), f32x16{});
    else acc = product(w, (l - 1) & 1);
    __bf16 v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      z[l][r] = acc[r] + s_b[l * HID + 32 * mb + crow(r, h)];
      v[r] = to_bf16(act(z[l][r]));
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) w[t] = wn[t];
    if (l < 2) fetch(A.W[l + 2], 8, wn);
    else if (l == 2) {
      // the output layer's 32 rows are one tile, wave 0's
#pragma unroll
      for (int t = 0; t < 8; ++t)
        wn[t] = *reinterpret_cast<const bf16x8*>(A.W[4] + (t * 64 + lane) * 8);
    } else if (A.backward) {
      fetch(A.WT[4], 1, wn);
    }
    emit(v, l & 1, A.act[l + 1], HID);
  }
  // outputs, and their errors 2 (Y - T) / (7 B) in place of the inputs
  if (mb == 0) {
    const f32x16 acc = product(w, 1);
    const int64_t b = tile * 32 + i;
    const float sc = 2.f / (7.f * float(A.B));
    __bf16 g[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 4 * h + r;
      const float t = s_T[i][k];
      const float y = k < NOUT ? acc[r] + s_b[4 * HID + k] : 0.f;
      if (A.Y) {
        A.Y[b * 8 + k] = y;
        A.T8[b * 8 + k] = t;
      }
      g[r] = to_bf16(k < NOUT ? sc * (y - t) : 0.f);
      s_x[i][k] = g[r];
      s_x[i][8 + k] = to_bf16(0.f);
      if (A.backward) A.err[4][((b >> 4) * 8 + k) * 16 + (b & 15)] = g[r];
    }
  }
  if (!A.backward) return;
  lds_barrier();
  bf16x8 wb[8];
  fetch(A.WT[3], 8, wb);
#pragma unroll
  for (int l = 3; l >= 0; --l) {
    // error at the output of layer l: W_{l+1}^T err_{l+1}, times a'(z_l)
    f32x16 acc;
    if (l == 3) acc = mfma(wn[0], *reinterpret_cast<const bf16x8*>(&s_x[i][8 * h]), f32x16{});
    else acc = product(w, (l + 1) & 1);
    __bf16 v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = to_bf16(acc[r] * act_grad(z[l][r]));
#pragma unroll
    for (int t = 0; t < 8; ++t) w[t] = wb[t];
    if (l >= 2) fetch(A.WT[l - 1], 8, wb);
    emit(v, l & 1, A.err[l], HID);
  }
}

// loss partial sums per 256 points
__global__ void __launch_bounds__(256) k_sur_loss(const float* __restrict__ Y,
                                                  const float* __restrict__ T, int B,
                                                  float* partial) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (b < B)
    for (int k = 0; k < 7; ++k) {
      const float diff = Y[int64_t(b) * 8 + k] - T[int64_t(b) * 8 + k];
      l += diff * diff;
    }
  __shared__ float sh[4];
  for (int o = 32; o > 0; o >>= 1) l += __shfl_down(l, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Weight and bias gradients of every layer, split over batch chunks, one wave
// per 32 x 32 tile and chunk:
//   partial[c][n][k]    = sum_{b in chunk c} err[n][b] act[k][b]   (k < act_rows)
//   partial[c][n][rows] = sum_{b in chunk c} err[n][b]             (bias)
// The points of a chunk are one chain of MFMAs (64 in chunks of 1,024), so the
// loads of the next group of 8 steps are in flight while the current one
// multiplies: bound by the operands' way from the L2.  The chunk is the fastest
// index of the waves, so that with 8 chunks each XCD reads one chunk only (9.6
// -> 9.0 us at a batch of 8,192, and the layers' separate launches before:
// 17 to 19.5 us each, 93 together).
struct WeightGradArgs {
  const __bf16* act[5];
  const __bf16* err[5];
  float* partial[5];
  int first[6];  // first wave of each layer
  int chunk, nch;
};
__host__ __device__ constexpr int grad_tiles(int layer) {
  return ((layer == 4 ? 32 : HID) / 32) * ((act_rows(layer) + 1 + 31) / 32);
}

template <int L>
__device__ __forceinline__ void weight_gradient_tile(const WeightGradArgs& A, int wave, int lane) {
  constexpr int MB = (L == 4 ? 32 : HID) / 32, KR = act_rows(L), ER = err_rows(L);
  constexpr int nout = L == 4 ? NOUT : HID, STEP = 8;
  const int ch = wave % A.nch, mb = (wave / A.nch) % MB, kb = wave / (A.nch * MB);
  const int i = lane & 31, h = lane >> 5;
  const int n_a = 32 * mb + i, k_b = 32 * kb + i;
  const int64_t g0 = int64_t(ch) * (A.chunk / 16);
  const bf16x8 zero = bf16x8{};
  bf16x8 one;
#pragma unroll
  for (int s = 0; s < 8; ++s) one[s] = to_bf16(1.f);
  const bool has_a = n_a < ER, has_b = k_b < KR;
  const bf16x8 fill = k_b == KR ? one : zero;
  const __bf16* pa = A.err[L] + (g0 * ER + (has_a ? n_a : 0)) * 16 + 8 * h;
  const __bf16* pb = A.act[L] + (g0 * KR + (has_b ? k_b : 0)) * 16 + 8 * h;
  bf16x8 a[STEP], b[STEP], an[STEP], bn[STEP];
  auto load = [&](int t, bf16x8 (&x)[STEP], bf16x8 (&y)[STEP]) {
#pragma unroll
    for (int s = 0; s < STEP; ++s) {
      x[s] = has_a ? *reinterpret_cast<const bf16x8*>(pa + int64_t(t + s) * ER * 16) : zero;
      y[s] = has_b ? *reinterpret_cast<const bf16x8*>(pb + int64_t(t + s) * KR * 16) : fill;
    }
  };
  const int steps = A.chunk / 16;  // 16 or 64
  f32x16 acc = f32x16{};
  load(0, a, b);
  for (int t = 0; t < steps; t += STEP) {
    if (t + STEP < steps) load(t + STEP, an, bn);
#pragma unroll
    for (int s = 0; s < STEP; ++s) acc = mfma(a[s], b[s], acc);
#pragma unroll
    for (int s = 0; s < STEP; ++s) {
      a[s] = an[s];
      b[s] = bn[s];
    }
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int n = 32 * mb + crow(v, h);
    if (n < nout && k_b <= KR) A.partial[L][(int64_t(ch) * nout + n) * (KR + 1) + k_b] = acc[v];
  }
}

__global__ void __launch_bounds__(64) k_sur_weight_gradients(WeightGradArgs A) {
  const int wave = blockIdx.x, lane = threadIdx.x;
  // the layer is uniform over the wave
  if (wave < A.first[1]) weight_gradient_tile<0>(A, wave, lane);
  else if (wave < A.first[2]) weight_gradient_tile<1>(A, wave - A.first[1], lane);
  else if (wave < A.first[3]) weight_gradient_tile<2>(A, wave - A.first[2], lane);
  else if (wave < A.first[4]) weight_gradient_tile<3>(A, wave - A.first[3], lane);
  else if (wave < A.first[5]) weight_gradient_tile<4>(A, wave - A.first[4], lane);
}

struct LayerDesc {
  int nout, nin, kc;     // kc: partial columns before the bias column (16 for layer 0)
  int off_w, off_b;
  const float* partial;  // [nch][nout][kc + 1]
  __bf16* W;             // fragments of the weights and, layers 1 to 4, of their transpose
  __bf16* WT;
  int first;             // first thread of the layer
};
struct UpdateArgs {
  LayerDesc layer[5];
  int threads;
};

// gradient of every parameter from the chunk partials (fixed order); then
// either an Adam step on the FP32 master copy (refreshing the BF16 copies) or
// a plain copy of the gradient to `grad_out`
__global__ void __launch_bounds__(256) k_sur_update(UpdateArgs U, int nch, float* params,
                                                    float* m1, float* m2, float lr, float beta1,
                                                    float beta2, float eps, float bc1, float bc2,
                                                    float* grad_out) {
  const int at = blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= U.threads) return;
  int l = 0;
#pragma unroll
  for (int k = 1; k < 5; ++k)
    if (at >= U.layer[k].first) l = k;
  const LayerDesc L = U.layer[l];
  const int idx = at - L.first;
  const int nw = L.nout * L.nin;
  const bool is_w = idx < nw;
  const int n = is_w ? idx / L.nin : idx - nw;
  const int k = is_w ? idx % L.nin : L.kc;
  const int cols = L.kc + 1;
  // layer 0: x_hi and x_lo share the weight, added after each chunk's x_hi
  const bool pair = is_w && L.kc == K0;
  float g = 0.f;
  for (int c = 0; c < nch; c += 4) {
    float p[4], q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float* P = L.partial + (int64_t(min(c + j, nch - 1)) * L.nout + n) * cols;
      p[j] = P[k];
      q[j] = pair ? P[k + NIN] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (c + j < nch) {
        g += p[j];
        if (pair) g += q[j];
      }
  }
  const int p = is_w ? L.off_w + idx : L.off_b + n;
  if (grad_out) {
    grad_out[p] = g;
    return;
  }
  const float a = beta1 * m1[p] + (1.f - beta1) * g;
  const float b = beta2 * m2[p] + (1.f - beta2) * g * g;
  m1[p] = a;
  m2[p] = b;
  const float w = params[p] - lr * (a / bc1) / (sqrtf(b / bc2) + eps);
  params[p] = w;
  if (is_w) {
    const __bf16 wb = to_bf16(w);
    const int ks = l == 0 ? 1 : 8;
    L.W[frag(n, k, ks)] = wb;
    if (l == 0) L.W[frag(n, k + NIN, ks)] = wb;
    else L.WT[frag(k, n, l == 4 ? 1 : 8)] = wb;
  }
}

// BF16 copies of the master weights (fragments, both orientations) and the
// permuted inference image, FP16 or (bf16 != 0) BF16
__global__ void __launch_bounds__(256) k_sur_refresh(const float* __restrict__ P, __bf16* W0,
                                                     __bf16* W1, __bf16* W2, __bf16* W3,
                                                     __bf16* W4, __bf16* T1, __bf16* T2,
                                                     __bf16* T3, __bf16* T4, f16x8* img,
                                                     float* imgb, int bf16) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  // forward / transposed copies
  if (idx < HID * K0) {
    const int n = idx / K0, k = idx % K0;
    const float w = k < NIN ? P[OFF_W0 + n * NIN + k] : k < 2 * NIN ? P[OFF_W0 + n * NIN + k - NIN] : 0.f;
    W0[frag(n, k, 1)] = to_bf16(w);
  }
  if (idx < HID * HID) {
    const int n = idx / HID, k = idx % HID;
    const __bf16 a = to_bf16(P[OFF_W1 + idx]), b = to_bf16(P[OFF_W2 + idx]),
                 c = to_bf16(P[OFF_W3 + idx]);
    const int f = frag(n, k, 8), ft = frag(k, n, 8);
    W1[f] = a; W2[f] = b; W3[f] = c;
    T1[ft] = a; T2[ft] = b; T3[ft] = c;
  }
  if (idx < 32 * HID) {
    const int n = idx / HID, k = idx % HID;
    const __bf16 w = to_bf16(n < NOUT ? P[OFF_W4 + n * HID + k] : 0.f);
    W4[frag(n, k, 8)] = w;
    if (n < 16) T4[frag(k, n, 1)] = w;
  }
  // permuted image: one thread per (vector, slot)
  if (idx < PW_SIZE * 8) {
    const int vec = idx / 8, s = idx % 8, lane = vec % 64, i = lane & 31, h = lane >> 5;
    float w = 0.f;
    if (vec < PW_L1) {
      const int mb = vec / 64, k = 8 * h + s, row = 32 * mb + i;
      w = k < NIN ? P[OFF_W0 + row * NIN + k] : k < 2 * NIN ? P[OFF_W0 + row * NIN + k - NIN] : 0.f;
    } else if (vec < PW_L4) {
      const int l = (vec - PW_L1) / (4 * 8 * 64), rem = (vec - PW_L1) % (4 * 8 * 64);
      const int mb = rem / (8 * 64), t = (rem / 64) % 8, row = 32 * mb + i;
      const int off = l == 0 ? OFF_W1 : l == 1 ? OFF_W2 : OFF_W3;
      w = P[off + row * HID + chain_k(t, h, s)];
    } else {
      const int t = (vec - PW_L4) / 64;
      w = i < NOUT ? P[OFF_W4 + i * HID + chain_k(t, h, s)] : 0.f;
    }
    if (bf16)
      reinterpret_cast<Bf16::x8*>(img)[vec][s] = static_cast<__bf16>(w);
    else
      img[vec][s] = static_cast<_Float16>(w);
  }
  if (idx < PB_SIZE) {
    float b = 0.f;
    if (idx < 4 * HID) {
      const int l = idx / HID, n = idx % HID;
      const int off = l == 0 ? OFF_B0 : l == 1 ? OFF_B1 : l == 2 ? OFF_B2 : OFF_B3;
      b = P[off + n];
    } else if (idx - 4 * HID < NOUT) {
      b = P[OFF_B4 + idx - 4 * HID];
    }
    imgb[idx] = b;
  }
}

// evaluation of the network on n points (scaled inputs, sx floats per point
// -> outputs, sy floats per point); persistent blocks of 8 or 12 waves, the image
// staged in LDS once per block.  With 8 floats per point on both sides (the
// explicit step's buffers) the points move as two 16-byte words and the 8th
// input float, the strain pass's envelope flag, is copied to the 8th output
// float, where the force pass reads it with the outputs.
template <class F>
__global__ void __launch_bounds__(768) k_sur_infer(const typename F::x8* __restrict__ img,
                                                   const float* __restrict__ imgb, int64_t n,
                                                   const float* __restrict__ X, int sx, float* Y,
                                                   int sy) {
  __shared__ Image<F> L;
  stage_image<F>(L, img, imgb);
  __syncthreads();
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int64_t tiles = (n + 31) / 32;
  const int waves = blockDim.x >> 6;
  const int64_t stride = int64_t(gridDim.x) * waves;
  const bool vec8 = sx == 8 && sy == 8;
  int64_t tile = int64_t(blockIdx.x) * waves + (threadIdx.x >> 6);
  // the next tile's inputs are loaded while the current one is evaluated;
  // lanes past the end read point 0 (n > 0) and use zeros
  float xn[8];
  auto load = [&](int64_t tl, float* x) {
    const int64_t p = tl * 32 + j;
    const bool ok = tl < tiles && p < n;
    const float* src = X + (ok ? p * sx : 0);
    float v[8];
    if (vec8) {
      const float4 a = reinterpret_cast<const float4*>(src)[0];
      const float4 b = reinterpret_cast<const float4*>(src)[1];
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
      for (int k = 0; k < 7; ++k) v[k] = src[k];
      v[7] = 0.f;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = ok ? v[k] : 0.f;
  };
  load(tile, xn);
  for (; tile < tiles; tile += stride) {
    float x[8], y[7];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = xn[k];
    load(tile + stride, xn);
    eval_wave<F>(L, x, y);
    const int64_t p = tile * 32 + j;
    if (p < n && h == 0) {
      if (vec8) {
        float4* dst = reinterpret_cast<float4*>(Y + p * 8);
        dst[0] = make_float4(y[0], y[1], y[2], y[3]);
        dst[1] = make_float4(y[4], y[5], y[6], x[7]);
      } else {
#pragma unroll
        for (int k = 0; k < 7; ++k) Y[p * sy + k] = y[k];
      }
    }
  }
}

template <typename T>
hipError_t dalloc_n(T** p, size_t n) {
  *p = nullptr;
  return hipMalloc(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T));
}
template <typename T>
void dfree_p(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

}  // namespace

// ---------------------------------------------------------------------------
Surrogate::~Surrogate() { release(); }

void Surrogate::release_batch() {
  dfree_p(Tb); dfree_p(Yb); dfree_p(loss_part);
  for (int l = 0; l < 5; ++l) { dfree_p(act[l]); dfree_p(err[l]); dfree_p(part[l]); }
  bcap = 0;
}

void Surrogate::release() {
  release_batch();
  dfree_p(params); dfree_p(m1); dfree_p(m2); dfree_p(grad);
  for (int l = 0; l < 5; ++l) { dfree_p(Wbf[l]); dfree_p(WT[l]); }
  dfree_p(img); dfree_p(imgb);
  dfree_p(X); dfree_p(T);
  dfree_p(fallbacks);
  dfree_p(io_x); dfree_p(io_y);
  dfree_p(pt_x); dfree_p(pt_y);
  nsamples = 0;
  io_cap = 0;
  pt_cap = 0;
}

hipError_t Surrogate::ensure_params() {
  if (params) return hipSuccess;
  hipError_t e;
  if ((e = dalloc_n(&params, NPARAM)) || (e = dalloc_n(&m1, NPARAM)) || (e = dalloc_n(&m2, NPARAM)) ||
      (e = dalloc_n(&grad, NPARAM)))
    return e;
  const int kbf[5] = {K0, HID, HID, HID, HID};
  const int rows[5] = {HID, HID, HID, HID, 32};
  for (int l = 0; l < 5; ++l)
    if ((e = dalloc_n(&Wbf[l], size_t(rows[l]) * kbf[l]))) return e;
  for (int l = 1; l < 5; ++l)
    if ((e = dalloc_n(&WT[l], size_t(HID) * (l == 4 ? 16 : HID)))) return e;
  if ((e = dalloc_n(&img, size_t(PW_SIZE) * 8)) || (e = dalloc_n(&imgb, PB_SIZE)) ||
      (e = dalloc_n(&fallbacks, 1)))
    return e;
  if ((e = hipMemset(fallbacks, 0, sizeof(unsigned long long)))) return e;
  // deterministic initialisation: U(-a, a), a = sqrt(3 / fan_in), zero biases
  std::vector<float> h(NPARAM, 0.f);
  std::mt19937_64 gen(0x5eed5eedull);
  auto fill = [&](int off, int nout, int nin) {
    const float a = std::sqrt(3.f / float(nin));
    std::uniform_real_distribution<float> U(-a, a);
    for (int k = 0; k < nout * nin; ++k) h[off + k] = U(gen);
  };
  fill(OFF_W0, HID, NIN);
  fill(OFF_W1, HID, HID);
  fill(OFF_W2, HID, HID);
  fill(OFF_W3, HID, HID);
  fill(OFF_W4, NOUT, HID);
  if ((e = hipMemcpy(params, h.data(), NPARAM * 4, hipMemcpyHostToDevice))) return e;
  if ((e = hipMemset(m1, 0, NPARAM * 4)) || (e = hipMemset(m2, 0, NPARAM * 4))) return e;
  for (int l = 1; l < 5; ++l)
    if ((e = hipMemset(WT[l], 0, size_t(HID) * (l == 4 ? 16 : HID) * 2))) return e;
  step = 0;
  return hipSuccess;
}

hipError_t Surrogate::refresh(hipStream_t s) {
  const int nthreads = std::max({HID * HID, PW_SIZE * 8});
  k_sur_refresh<<<(nthreads + 255) / 256, 256, 0, s>>>(params, Wbf[0], Wbf[1], Wbf[2], Wbf[3],
                                                       Wbf[4], WT[1], WT[2], WT[3], WT[4], img,
                                                       imgb, int(infer_bf16));
  return hipGetLastError();
}

hipError_t Surrogate::ensure_batch(int B) {
  if (B <= bcap) return hipSuccess;
  release_batch();
  hipError_t e;
  const size_t b = size_t(B);
  if ((e = dalloc_n(&Tb, b * 8)) || (e = dalloc_n(&Yb, b * 8)) ||
      (e = dalloc_n(&loss_part, (b + 255) / 256)))
    return e;
  // chunk partials: at most B / 256 chunks of [nout][kc + 1]
  const size_t nch = b / 256;
  for (int l = 0; l < 5; ++l)
    if ((e = dalloc_n(&act[l], b * act_rows(l))) || (e = dalloc_n(&err[l], b * err_rows(l))) ||
        (e = dalloc_n(&part[l], nch * (l == 4 ? NOUT : HID) * (act_rows(l) + 1))))
      return e;
  bcap = B;
  return hipSuccess;
}

// k_sur_pass on a batch of B samples of (x, t): drawn for iteration `iter`
// (iter >= 0) or the first B
hipError_t Surrogate::run_pass(hipStream_t s, const float* x, const float* t, int64_t n, int B,
                               uint64_t seed, int64_t iter, bool backward, bool outputs) {
  PassArgs A;
  A.X = x;
  A.T = t;
  A.n = n;
  A.B = B;
  A.seed = seed;
  A.iter = iter < 0 ? 0 : iter;
  A.draw = iter >= 0;
  for (int l = 0; l < 5; ++l) {
    A.W[l] = Wbf[l];
    A.WT[l] = WT[l];
    A.act[l] = act[l];
    A.err[l] = err[l];
  }
  A.params = params;
  A.Y = outputs ? Yb : nullptr;
  A.T8 = Tb;
  A.backward = backward;
  k_sur_pass<<<unsigned(B / 32), 256, 0, s>>>(A);
  return hipGetLastError();
}

// parameter gradients of the batch that k_sur_pass went back through; then
// either an Adam step (grad_only = false) or the gradient into `grad`
// (grad_only = true)
hipError_t Surrogate::apply(hipStream_t s, int B, bool grad_only, float lr) {
  const int chunk = (B % 1024 == 0) ? 1024 : 256;
  const int nch = B / chunk;
  WeightGradArgs G;
  G.chunk = chunk;
  G.nch = nch;
  G.first[0] = 0;
  for (int l = 0; l < 5; ++l) {
    G.act[l] = act[l];
    G.err[l] = err[l];
    G.partial[l] = part[l];
    G.first[l + 1] = G.first[l] + grad_tiles(l) * nch;
  }
  k_sur_weight_gradients<<<unsigned(G.first[5]), 64, 0, s>>>(G);
  hipError_t e = hipGetLastError();
  if (e) return e;
  const int offw[5] = {OFF_W0, OFF_W1, OFF_W2, OFF_W3, OFF_W4};
  const int offb[5] = {OFF_B0, OFF_B1, OFF_B2, OFF_B3, OFF_B4};
  const float b1 = 0.9f, b2 = 0.999f;
  if (!grad_only) ++step;
  const float bc1 = 1.f - std::pow(b1, float(std::max<int64_t>(step, 1)));
  const float bc2 = 1.f - std::pow(b2, float(std::max<int64_t>(step, 1)));
  UpdateArgs U;
  U.threads = 0;
  for (int l = 0; l < 5; ++l) {
    LayerDesc& L = U.layer[l];
    L.nout = l == 4 ? NOUT : HID;
    L.nin = l == 0 ? NIN : HID;
    L.kc = act_rows(l);
    L.off_w = offw[l];
    L.off_b = offb[l];
    L.partial = part[l];
    L.W = Wbf[l];
    L.WT = WT[l];
    L.first = U.threads;
    U.threads += L.nout * L.nin + L.nout;
  }
  k_sur_update<<<(U.threads + 255) / 256, 256, 0, s>>>(U, nch, params, m1, m2, lr, b1, b2, 1e-8f,
                                                       bc1, bc2, grad_only ? grad : nullptr);
  return hipGetLastError();
}

hipError_t Surrogate::generate(hipStream_t s, int64_t paths, int steps, double inc_std,
                               double yd_scale, double yd_shape, uint64_t seed) {
  dfree_p(X);
  dfree_p(T);
  nsamples = 0;
  const int64_t n = paths * steps;
  hipError_t e;
  if ((e = dalloc_n(&X, size_t(n) * 7)) || (e = dalloc_n(&T, size_t(n) * 7))) return e;
  k_sur_gen<<<unsigned((paths + 255) / 256), 256, 0, s>>>(paths, steps, eps, inc_std, lambda, mu,
                                                          Sd, yd_scale, yd_shape, sS, sW, seed, X, T);
  if ((e = hipGetLastError())) return e;
  nsamples = n;
  return hipSuccess;
}

hipError_t Surrogate::train(hipStream_t s, int iterations, int B, double lr0, uint64_t seed,
                            double* final_loss) {
  hipError_t e;
  if ((e = ensure_params()) || (e = ensure_batch(B))) return e;
  if ((e = refresh(s))) return e;
  const int warm = std::min(200, iterations / 10 + 1);
  double loss = 0;
  for (int it = 0; it < iterations; ++it) {
    // linear warm-up, then cosine decay to lr0 / 100
    double lr = lr0;
    if (it < warm) lr = lr0 * double(it + 1) / warm;
    else lr = lr0 * (0.01 + 0.99 * 0.5 * (1 + std::cos(M_PI * double(it - warm) /
                                                      double(std::max(1, iterations - warm)))));
    if ((e = run_pass(s, X, T, nsamples, B, seed, it, true, false)) ||
        (e = apply(s, B, false, float(lr))))
      return e;
  }
  if ((e = refresh(s))) return e;
  // loss of the last batch (after the final update, on the same batch)
  if ((e = run_pass(s, X, T, nsamples, B, seed, iterations - 1, false, true)) ||
      (e = batch_loss(s, B, &loss)))
    return e;
  if (final_loss) *final_loss = loss;
  return hipSuccess;
}

// mean squared error of the outputs that the last pass wrote
hipError_t Surrogate::batch_loss(hipStream_t s, int B, double* loss) {
  const int nb = (B + 255) / 256;
  k_sur_loss<<<nb, 256, 0, s>>>(Yb, Tb, B, loss_part);
  hipError_t e = hipGetLastError();
  if (e) return e;
  std::vector<float> h(nb);
  if ((e = hipMemcpyAsync(h.data(), loss_part, nb * 4, hipMemcpyDeviceToHost, s)) ||
      (e = hipStreamSynchronize(s)))
    return e;
  double sum = 0;
  for (float v : h) sum += v;
  *loss = sum / (7.0 * B);
  return hipSuccess;
}

hipError_t Surrogate::gradients(hipStream_t s, int device, HostCopier& copy, int64_t n,
                                const float* x_host, const float* t_host, float* grad_host,
                                double* loss) {
  hipError_t e;
  const int B = int(n);
  if ((e = ensure_params()) || (e = ensure_batch(B)) || (e = ensure_io(n))) return e;
  if ((e = refresh(s))) return e;
  float* tdev = io_y;
  if ((e = copy.to_device(device, s, io_x, x_host, size_t(n) * 7 * 4)) ||
      (e = copy.to_device(device, s, tdev, t_host, size_t(n) * 7 * 4)))
    return e;
  if ((e = run_pass(s, io_x, tdev, n, B, 0, -1, true, true)) || (e = apply(s, B, true, 0.f)))
    return e;
  if ((e = copy.to_host(device, s, grad_host, grad, NPARAM * 4))) return e;
  return batch_loss(s, B, loss);
}

hipError_t Surrogate::ensure_io(int64_t n) {
  if (n <= io_cap) return hipSuccess;
  dfree_p(io_x);
  dfree_p(io_y);
  hipError_t e;
  if ((e = dalloc_n(&io_x, size_t(n) * 7)) || (e = dalloc_n(&io_y, size_t(n) * 7))) return e;
  io_cap = n;
  return hipSuccess;
}

hipError_t Surrogate::infer(hipStream_t s, int device, HostCopier& copy, int64_t n,
                            const float* x_host, float* y_host) {
  hipError_t e;
  if ((e = ensure_params()) || (e = ensure_io(n))) return e;
  if ((e = copy.to_device(device, s, io_x, x_host, size_t(n) * 7 * 4))) return e;
  if ((e = launch_sur_mlp(s, img, imgb, infer_bf16, n, io_x, 7, io_y, 7))) return e;
  return copy.to_host(device, s, y_host, io_y, size_t(n) * 7 * 4);
}

hipError_t launch_sur_mlp(hipStream_t s, const void* img, const float* imgb, bool bf16,
                          int64_t n, const float* x, int sx, float* y, int sy) {
  (void)hipGetLastError();
  if (n <= 0) return hipSuccess;
  // One block per CU (the weight image fills most of the LDS), so that one
  // wave's activations overlap another's MFMAs: 8 waves, or 12 where they take
  // less than three quarters as many rounds of a tile per wave (a round of 12
  // takes about 4/3 of one of 8).  Step of a plate with the network, 8 / 12
  // waves: 77,568 points 32.1 / 28.6 us (2 rounds, 1), 112,752 34.0 / 37.8 (2,
  // 2), 160,320 42.9 / 40.7 (3, 2), 4.03 M 587 / 578 (62, 42), where 12 reach
  // 1.04 PFLOP/s.
  const int64_t tiles = (n + 31) / 32;
  auto rounds = [&](int waves) { return (tiles + CARD_CUS * waves - 1) / (CARD_CUS * waves); };
  const int waves = rounds(12) * 4 < rounds(8) * 3 ? 12 : 8;
  const unsigned g = unsigned(std::min<int64_t>(CARD_CUS, (tiles + waves - 1) / waves));
  if (bf16)
    k_sur_infer<Bf16><<<g, 64 * waves, 0, s>>>(static_cast<const Bf16::x8*>(img), imgb, n, x, sx,
                                               y, sy);
  else
    k_sur_infer<Fp16><<<g, 64 * waves, 0, s>>>(static_cast<const Fp16::x8*>(img), imgb, n, x, sx,
                                               y, sy);
  return hipGetLastError();
}

hipError_t Surrogate::ensure_points(int64_t n) {
  if (n <= pt_cap) return hipSuccess;
  dfree_p(pt_x);
  dfree_p(pt_y);
  hipError_t e;
  if ((e = dalloc_n(&pt_x, size_t(n) * 8)) || (e = dalloc_n(&pt_y, size_t(n) * 8))) return e;
  pt_cap = n;
  return hipSuccess;
}

hipError_t Surrogate::set_params(hipStream_t s, const float* host) {
  hipError_t e;
  if ((e = ensure_params())) return e;
  if ((e = hipMemcpyAsync(params, host, NPARAM * 4, hipMemcpyHostToDevice, s))) return e;
  if ((e = hipMemsetAsync(m1, 0, NPARAM * 4, s)) || (e = hipMemsetAsync(m2, 0, NPARAM * 4, s)))
    return e;
  step = 0;
  if ((e = refresh(s))) return e;
  return hipStreamSynchronize(s);
}

hipError_t Surrogate::get_params(hipStream_t s, float* host) {
  hipError_t e;
  if ((e = ensure_params())) return e;
  if ((e = hipMemcpyAsync(host, params, NPARAM * 4, hipMemcpyDeviceToHost, s))) return e;
  return hipStreamSynchronize(s);
}

}  // namespace akx
