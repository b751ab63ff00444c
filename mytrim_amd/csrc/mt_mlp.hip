// Training and evaluation kernels of the scattering surrogate (mt_mlp.h).
//
//   mlp_data      training pairs sampled as the cascade samples (eps, b),
//                 or on a rectangle in (log eps, b); target ln s2 from
//                 scatter_stable<double> (universal potential), one Philox
//                 stream per sample
//   mlp_pass      forward and backward pass on the matrix cores
//   mlp_grad      gradient and loss of chunks of 128 samples, matrix cores
//   mlp_update    the chunks' sums added in order (deterministic, no atomics)
//                 and the Adam update with a cosine step-size schedule
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "mt_mlp.h"
#include "mt_philox.h"
#include "mt_physics.h"

namespace mt {

// maximum impact parameter of a triple at flight energy E (trim.C:88-95)
__device__ __forceinline__ double mlp_pmax(const MlpTriple& t, double E) {
  const double eeg = sqrt(E * t.f * t.epsdg);
  return t.a / (eeg + sqrt(eeg) + 0.125 * pow(eeg, 0.1));
}

// Training pairs, one Philox stream per sample; labels from the FP64 MAGIC
// solve.  Two samplings:
//   rect = 0: the way the cascade draws them: a random triple, a flight
//             energy (half log-uniform, half uniform on [E_lo, E_hi of the
//             triple]), eps = fi E and b = pmax(E) sqrt(u) / ai;
//   rect = 1: a rectangle: eps log-uniform on [eps_lo, eps_hi], b uniform on
//             [0, b_hi].
__global__ void __launch_bounds__(256) mlp_data(uint32_t seed, long long n, const MlpTriple* tri, int n_tri,
                                                double E_lo, int rect, double eps_lo, double eps_hi, double b_hi,
                                                MlpNorm nm, float* X, float* T, float* m, float* v, int* t) {
  // the optimiser's state starts at zero
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < kMlpParams; i += gridDim.x * blockDim.x) {
    m[i] = 0.0f;
    v[i] = 0.0f;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *t = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const P4 r = philox10((uint32_t)i, (uint32_t)(i >> 32), 0x5a17u, 0u, seed, 0x6d6c70u);
    const P4 r2 = philox10((uint32_t)i, (uint32_t)(i >> 32), 0x5a18u, 0u, seed, 0x6d6c70u);
    const double u = u53(r.y, r.z);
    double eps, b;
    if (rect) {
      eps = eps_lo * pow(eps_hi / eps_lo, u);
      b = b_hi * u32d(r.w);
    } else {
      const int k = min((int)(u32d(r.x) * n_tri), n_tri - 1);
      const MlpTriple t = tri[k];
      const double E = (r2.x & 1u) ? E_lo * pow(t.E_hi / E_lo, u) : E_lo + (t.E_hi - E_lo) * u;
      eps = t.fi * E;
      b = mlp_pmax(t, E) * sqrt(u32d(r.w)) / t.ai;
    }
    double s2, ct, st;
    int it;
    scatter_stable<double, 0>(eps, b, s2, ct, st, it);
    float x0, x1, x2;
    mlp_inputs(nm, (float)eps, (float)b, x0, x1, x2);
    X[3 * i] = x0;
    X[3 * i + 1] = x1;
    X[3 * i + 2] = x2;
    T[i] = (float)((log(fmax(s2, 1e-300)) - nm.y_off) / nm.y_scale);
  }
}

// Loss and gradient of one batch in two kernels.  The products run on the matrix
// cores in single precision, as 16 x 16 tiles of v_mfma_f32_16x16x4_f32.  Layout
// of that instruction (lane l, n = l % 16, q = l / 16): A[n][q], B[q][n],
// D[4 q + r][n]; it adds its four products one after another, each a fused
// multiply-add, so step c with the inner indices 4 c + q gives the sums of a
// serial loop bit for bit.
//
// mlp_pass: forward and backward pass of 16 samples per block (256 blocks for a
// batch of 4096): z2 = h1 W2^T, y = h2 W3, g1 = d2 W2, a wave per 16 columns.
// The activations and deltas go to `rec` ([h1 | d1 | h2 | d2][S][64], then dy[S]
// and e^2[S], S the batch rounded up to whole chunks, then 1 and 0; activations and
// deltas of the samples past the batch are zero, whatever the weights: 0 times an
// infinite one would reach the sums).
// mlp_grad: sums of delta x input over a chunk of 128 samples, a wave per 16 x 16
// tile of a weight matrix, into part[chunk][kMlpParams + 1] (the last entry: the
// squared errors).
// A step of 4096 took 60 + 39 us with one lane per sample (16 blocks, weights as
// scalars) and per parameter, and 24 us with both passes of a chunk in one block
// (32 of 256 CUs busy); these kernels take 6.5 and 4.6 us, mostly the latency of
// first touches and of the chain of layers.
// W2 rows are 80 floats apart in LDS, samples 68: the four q rows of a read fall
// in different banks.
constexpr int kTile = 16, kChunk = 128;
constexpr int kW2s = 80, kHs = 68;
typedef float mt_f32x4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256) mlp_pass(const float* __restrict__ p, const float* X, const float* T,
                                                long long base, int B, int S, int* t, float* rec) {
  __shared__ __align__(16) float w2[kMlpH * kW2s];
  __shared__ __align__(16) float h1[kTile * kHs], h2[kTile * kHs], d2[kTile * kHs];
  __shared__ float xs[kMlpIn][kTile], dys[kTile];
  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, n = l & 15, q = l >> 4;
  const int s0 = blockIdx.x * kTile, col = 16 * w + n;
  float* const rh1 = rec;
  float* const rd1 = rh1 + (size_t)S * kMlpH;
  float* const rh2 = rd1 + (size_t)S * kMlpH;
  float* const rd2 = rh2 + (size_t)S * kMlpH;
  float* const rdy = rd2 + (size_t)S * kMlpH;
  if (blockIdx.x == 0 && tid == 0) {
    if (t) *t += 1;  // steps begun: the update of this step reads it
    rdy[2 * (size_t)S] = 1.0f;
    rdy[2 * (size_t)S + 1] = 0.0f;
  }
  // every load of the block in one go: the weights were written by the last
  // update, so each first touch goes past this XCD's L2, over a microsecond
  float wl[16], w3q[16], tq[4];
#pragma unroll
  for (int i = 0; i < 16; ++i) wl[i] = p[kOffW2 + 256 * i + tid];
  const float f[4] = {p[kOffW1 + 3 * l], p[kOffW1 + 3 * l + 1], p[kOffW1 + 3 * l + 2], p[kOffB1 + l]};
  const float b2 = p[kOffB2 + col], w3 = p[kOffW3 + col], b3 = p[kOffB3];
  const int xi = tid < kMlpIn * kTile ? tid : 0;
  const float xv = s0 + xi / kMlpIn < B ? X[kMlpIn * (base + s0) + xi] : 0.0f;
#pragma unroll
  for (int c = 0; c < 16; ++c) w3q[c] = p[kOffW3 + 4 * c + q];
#pragma unroll
  for (int r = 0; r < 4; ++r) tq[r] = s0 + 4 * q + r < B ? T[base + s0 + 4 * q + r] : 0.0f;
  xs[xi % kMlpIn][xi / kMlpIn] = xv;
#pragma unroll
  for (int i = 0; i < 16; ++i) w2[(4 * i + w) * kW2s + l] = wl[i];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // layer 1 (mlp_h1): unit l of samples 4 w + r
    const int sm = 4 * w + r;
    const float t1 = mlp_tanh(f[0] * xs[0][sm] + f[1] * xs[1][sm] + f[2] * xs[2][sm] + f[3]);
    const float h = s0 + sm < B ? t1 : 0.0f;
    h1[sm * kHs + l] = h;
    rh1[(size_t)(s0 + sm) * kMlpH + l] = h;
  }
  __syncthreads();
  mt_f32x4 z = {b2, b2, b2, b2};  // layer 2: samples 4 q + r, unit col
#pragma unroll
  for (int c = 0; c < 16; ++c)
    z = __builtin_amdgcn_mfma_f32_16x16x4f32(h1[n * kHs + 4 * c + q], w2[col * kW2s + 4 * c + q], z, 0, 0, 0);
  float h2r[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    h2r[r] = s0 + 4 * q + r < B ? mlp_tanh(z[r]) : 0.0f;
    h2[(4 * q + r) * kHs + col] = h2r[r];
    rh2[(size_t)(s0 + 4 * q + r) * kMlpH + col] = h2r[r];
  }
  __syncthreads();
  if (w == 0) {  // layer 3: column 0 of the tile
    mt_f32x4 y = {b3, b3, b3, b3};
#pragma unroll
    for (int c = 0; c < 16; ++c)
      y = __builtin_amdgcn_mfma_f32_16x16x4f32(h2[n * kHs + 4 * c + q], n == 0 ? w3q[c] : 0.0f, y, 0, 0, 0);
    if (n == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int sm = 4 * q + r;
        const float e = s0 + sm < B ? y[r] - tq[r] : 0.0f;
        const float dy = 2.0f * e / (float)B;  // d(mean squared error)/dy
        dys[sm] = dy;
        rdy[s0 + sm] = dy;
        rdy[S + s0 + sm] = e * e;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float d = s0 + 4 * q + r < B ? dys[4 * q + r] * w3 * (1.0f - h2r[r] * h2r[r]) : 0.0f;
    d2[(4 * q + r) * kHs + col] = d;
    rd2[(size_t)(s0 + 4 * q + r) * kMlpH + col] = d;
  }
  __syncthreads();
  mt_f32x4 g = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < 16; ++c)
    g = __builtin_amdgcn_mfma_f32_16x16x4f32(d2[n * kHs + 4 * c + q], w2[(4 * c + q) * kW2s + col], g, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float h = h1[(4 * q + r) * kHs + col];
    rd1[(size_t)(s0 + 4 * q + r) * kMlpH + col] = s0 + 4 * q + r < B ? g[r] * (1.0f - h * h) : 0.0f;
  }
}

// a chunk's 29 tiles: 16 of dW2, 4 of (dW1 | db1), 4 of db2, 4 of dW3, one of
// (db3, loss)
constexpr int kGradTiles = 29;

__global__ void __launch_bounds__(256) mlp_grad(const float* X, const float* rec, long long base, int B, int S,
                                                float* part) {
  const int l = threadIdx.x & 63, n = l & 15, q = l >> 4;
  const int task = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), chunk = blockIdx.x;
  if (task >= kGradTiles) return;
  const float* const rh1 = rec;
  const float* const rd1 = rh1 + (size_t)S * kMlpH;
  const float* const rh2 = rd1 + (size_t)S * kMlpH;
  const float* const rd2 = rh2 + (size_t)S * kMlpH;
  const float* const rdy = rd2 + (size_t)S * kMlpH;
  const float* const one = rdy + 2 * (size_t)S;  // 1, 0
  // sample s's operands lie at a[s * as] and b[min(s, last) * bs]: a tile's
  // columns without an input read the constants
  const int kind = task < 16 ? 0 : task < 20 ? 1 : task < 24 ? 2 : task < 28 ? 3 : 4;
  const int ti = kind == 0 ? task >> 2 : task & 3;  // unit tile
  const size_t s0 = (size_t)chunk * kChunk;
  const float* a = (kind == 0 || kind == 2 ? rd2 : kind == 1 ? rd1 : rh2) + s0 * kMlpH + 16 * ti + n;
  const float* b = one + (n == (kind == 1 ? 3 : 0) ? 0 : 1);
  int as = kMlpH, bs = 0, last = kChunk - 1;
  if (kind == 0) {
    b = rh1 + s0 * kMlpH + 16 * (task & 3) + n;
    bs = kMlpH;
  } else if (kind == 1) {
    last = min(last, B - 1 - (int)s0);  // deltas past the batch are zero
    if (n < kMlpIn) {
      b = X + kMlpIn * (base + (long long)s0) + n;
      bs = kMlpIn;
    }
  } else if (kind == 3 && n == 0) {
    b = rdy + s0;
    bs = 1;
  } else if (kind == 4) {
    a = n < 2 ? rdy + n * (size_t)S + s0 : one + 1;
    as = n < 2 ? 1 : 0;
  }
  float fa[kChunk / 4], fb[kChunk / 4];
#pragma unroll
  for (int c = 0; c < kChunk / 4; ++c) {
    fa[c] = a[(4 * c + q) * as];
    fb[c] = b[min(4 * c + q, last) * bs];
  }
  mt_f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < kChunk / 4; ++c) d = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c], fb[c], d, 0, 0, 0);
  float* const out = part + (size_t)chunk * (kMlpParams + 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int u = 16 * ti + 4 * q + r;
    if (kind == 0) {
      out[kOffW2 + kMlpH * u + 16 * (task & 3) + n] = d[r];
    } else if (kind == 1) {
      if (n < kMlpIn) out[kOffW1 + kMlpIn * u + n] = d[r];
      if (n == 3) out[kOffB1 + u] = d[r];
    } else if (n == 0) {
      if (kind == 2) out[kOffB2 + u] = d[r];
      if (kind == 3) out[kOffW3 + u] = d[r];
      if (kind == 4 && q == 0 && r < 2) out[r == 0 ? kOffB3 : kMlpParams] = d[r];
    }
  }
}

// The chunks' sums added in order (deterministic, no atomics) and, with ADAM,
// the update (Kingma & Ba 2015, beta1 0.9, beta2 0.999; the step size follows a
// cosine from lr0 down to lr0 / 100; *t is the step).  One lane per parameter,
// its loads in flight together: latency bounds it.
template <bool ADAM>
__global__ void __launch_bounds__(64) mlp_update(const float* part, int n_parts, int B, float* g, float* loss_slot,
                                                 float* p, float* m, float* v, const int* t, float lr0,
                                                 int total_steps) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i > kMlpParams) return;
  float acc = 0.0f;
#pragma unroll 16
  for (int k = 0; k < n_parts; ++k) acc += part[(size_t)k * (kMlpParams + 1) + i];
  if (i == kMlpParams) {
    *loss_slot = acc / (float)B;
    return;
  }
  if constexpr (ADAM) {
    const int step = *t;
    const float b1 = 0.9f, b2 = 0.999f;
    const float frac = fminf((float)step / (float)total_steps, 1.0f);
    const float lr = lr0 * (0.01f + 0.495f * (1.0f + cosf(3.14159265f * frac)));
    m[i] = fmaf(b1, m[i], (1.0f - b1) * acc);
    v[i] = fmaf(b2, v[i], (1.0f - b2) * acc * acc);
    const float mh = m[i] / (1.0f - powf(b1, (float)step));
    const float vh = v[i] / (1.0f - powf(b2, (float)step));
    p[i] -= lr * mh / (sqrtf(vh) + 1e-8f);
  } else {
    g[i] = acc;
  }
}

__global__ void __launch_bounds__(256) mlp_infer(MlpDev S, const double* eps, const double* b, long long n,
                                                 double* s2) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const float v = mlp_s2(S, (float)eps[i], (float)b[i]);
    s2[i] = v < 0.0f ? -1.0 : (double)v;
  }
}

__global__ void mlp_pack_bf16(const float* p, uint32_t* w2bf) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < 64 * 32) {
    const int k = q / 32, jp = q % 32;
    w2bf[q] = bf16_bits(p[kOffW2 + 64 * k + 2 * jp]) | (bf16_bits(p[kOffW2 + 64 * k + 2 * jp + 1]) << 16);
  }
}

// ------------------------------------------------------------------ host side
static int grid_of(long long n) { return (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536); }

hipError_t mlp_make_data(uint32_t seed, long long n, const MlpTriple* tri, int n_tri, double E_lo, int rect,
                         const MlpNorm& nm, float* X, float* T, float* m, float* v, int* t, hipStream_t st) {
  hipLaunchKernelGGL(mlp_data, dim3(grid_of(n)), dim3(256), 0, st, seed, n, tri, n_tri, E_lo, rect,
                     (double)nm.eps_lo, (double)nm.eps_hi, (double)nm.b_hi, nm, X, T, m, v, t);
  return hipGetLastError();
}

// chunks of a batch of B: rows of its partial sums (kMlpParams + 1 floats each)
int mlp_parts(int B) { return (B + kChunk - 1) / kChunk; }
// floats of the batch's activations and deltas
size_t mlp_rec_floats(int B) { return (size_t)mlp_parts(B) * kChunk * (4 * kMlpH + 2) + 2; }

static void grad_launch(const float* p, const float* X, const float* T, long long base, int B, int* t, float* rec,
                        float* part, hipStream_t st) {
  const int parts = mlp_parts(B), S = parts * kChunk;
  hipLaunchKernelGGL(mlp_pass, dim3(S / kTile), dim3(256), 0, st, p, X, T, base, B, S, t, rec);
  hipLaunchKernelGGL(mlp_grad, dim3(parts, (kGradTiles + 3) / 4), dim3(256), 0, st, X, rec, base, B, S, part);
}

static void step_launch(float* p, const float* X, const float* T, long long base, int B, float* rec, float* part,
                        float* m, float* v, int* t, float lr0, int total, float* loss_slot, hipStream_t st) {
  grad_launch(p, X, T, base, B, t, rec, part, st);
  hipLaunchKernelGGL(mlp_update<true>, dim3((kMlpParams + 1 + 63) / 64), dim3(64), 0, st, part, mlp_parts(B), B,
                     nullptr, loss_slot, p, m, v, t, lr0, total);
}

// Train for `epochs` over n samples in batches of B (*t and the moments start
// at zero); losses[e] = mean batch loss of epoch e.  Several epochs replay one
// captured as a graph; a single one is launched directly (capturing and
// instantiating its nodes takes longer than launching them once).
hipError_t mlp_train(float* p, const float* X, const float* T, long long n, int B, int epochs, float lr0, float* rec, float* part,
                     float* m, float* v, int* t, float* batch_loss, double* losses, hipStream_t st) {
  const int steps = (int)(n / B);
  if (steps < 1) return hipErrorInvalidValue;
  const int total = steps * epochs;
  auto epoch = [&] {
    for (int s = 0; s < steps; ++s)
      step_launch(p, X, T, (long long)s * B, B, rec, part, m, v, t, lr0, total, batch_loss + s, st);
  };
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipError_t e = hipSuccess;
  if (epochs > 1) {
    e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    epoch();
    e = hipStreamEndCapture(st, &graph);
    if (e != hipSuccess) return e;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  }
  std::vector<float> bl(steps);
  for (int ep = 0; ep < epochs && e == hipSuccess; ++ep) {
    if (exec) {
      e = hipGraphLaunch(exec, st);
    } else {
      epoch();
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(bl.data(), batch_loss, steps * sizeof(float), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    double acc = 0.0;
    for (float x : bl) acc += x;
    losses[ep] = acc / steps;
  }
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  return e;
}

// gradient and loss of one batch (for checks against the CPU)
hipError_t mlp_batch_grad(const float* p, const float* X, const float* T, int B, float* rec, float* part, float* g,
                          float* loss, hipStream_t st) {
  grad_launch(p, X, T, 0ll, B, nullptr, rec, part, st);
  hipLaunchKernelGGL(mlp_update<false>, dim3((kMlpParams + 1 + 63) / 64), dim3(64), 0, st, part, mlp_parts(B), B, g,
                     loss, nullptr, nullptr, nullptr, nullptr, 0.0f, 1);
  return hipGetLastError();
}

hipError_t mlp_pack(const float* p, uint32_t* w2bf, hipStream_t st) {
  hipLaunchKernelGGL(mlp_pack_bf16, dim3(8), dim3(256), 0, st, p, w2bf);
  return hipGetLastError();
}

hipError_t mlp_infer_launch(const MlpDev& S, const double* eps, const double* b, long long n, double* s2,
                            hipStream_t st) {
  hipLaunchKernelGGL(mlp_infer, dim3(grid_of(n)), dim3(256), 0, st, S, eps, b, n, s2);
  return hipGetLastError();
}

}  // namespace mt
