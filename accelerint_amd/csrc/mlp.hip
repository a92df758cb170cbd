// Learned Newton start: BF16-MFMA training and inference kernels and the
// network's host-side owner (see mlp.hpp).  No counterpart in the reference.
//
// Training: mean squared error over normalized stage targets, Adam, batches of
// B samples (B a multiple of 16).  Two kernels per batch: k_mlp_rows runs the
// forward pass and the activations' gradients of 16 samples per block, row
// local from the gathered sample to dZ1; k_mlp_weights forms one 16x16 tile of
// a weight gradient per wavefront (or 16 bias gradients) over the whole batch
// and applies Adam to it at once.  Matrix operands are rounded to BF16 (nearest
// even) and accumulated in FP32 by v_mfma_f32_16x16x16_bf16, 16 values of the
// summed index per instruction in ascending order.
//
// What bounds it: launches and the latency of a short dependent chain -- a batch
// of 512 is 0.14 GFLOP and ~2 MB of traffic.  As one kernel per product and
// elementwise pass with the loss read back after every batch (17 launches, a copy
// and a device synchronization) a batch took 340 us; it takes 22 us now (two
// epochs of 32768 samples from host arrays: 44.0 -> 4.3 ms, parameters and losses
// bit-identical).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <random>
#include <string>
#include <vector>

#include "accelerint.h"
#include "mlp.hpp"

namespace acc {

// Device buffers of one batch (B samples, KT = B / 16 row tiles).  "Fragments"
// hold BF16 matrix tiles as the MFMA operands want them with the samples as the
// summed index: tile (row tile kt, column tile ct) lane l holds
// M[16 kt + 4 (l / 16) + i][16 ct + l % 16], i = 0..3, at ((ct * KT + kt) * 64 + l).
// That is also the layout of an MFMA result, so k_mlp_rows stores its result
// registers as they are and k_mlp_weights streams them without a transpose.
struct MlpBatch {
  const float* x;    // samples, row stride `in`
  const float* t;    // targets, row stride `out` (null: forward only)
  const int* idx;    // sample rows of the batch (null: 0, 1, ...)
  int in, inp, out, outp, rows;
  // weights: BF16 B-operand tiles of W1, W2, W3 and of W2^T, W3^T; FP32 biases
  const uint16_t *w1, *w2, *w3, *w2t, *w3t;
  const float *b1, *b2, *b3;
  // results
  float* y;          // [rows][out] (forward only)
  double* loss;      // squared error per row tile
  mlp_bf16x4 *fx, *fa1, *fa2, *fdy, *fdz2, *fdz1;  // fragments
  float *dy, *dz2, *dz1;                           // FP32 row-major (bias gradients)
};

constexpr int kMlpPad = 8;  // BF16 values between LDS rows: 16-byte rows, no bank pattern

// Operand tiles (0 .. kts - 1, kts <= KTS) of column tile nt of a weight matrix,
// in registers.
template <int KTS>
struct MlpW {
  mlp_bf16x4 b[KTS];
  __device__ __forceinline__ void load(const uint16_t* W, int nt, int kts) {
    const mlp_bf16x4* p = reinterpret_cast<const mlp_bf16x4*>(W) + (size_t)nt * kts * 64 + (threadIdx.x & 63);
#pragma unroll
    for (int kt = 0; kt < KTS; ++kt)
      if (kt < kts) b[kt] = p[(size_t)kt * 64];
  }
};
// D tile (16 samples x 16 columns) of A B: A from LDS rows (BF16, leading
// dimension lda).
template <int KTS>
__device__ __forceinline__ mlp_f32x4 mlp_tile(const uint16_t* A, int lda, const MlpW<KTS>& w, int kts) {
  const int l = (int)(threadIdx.x & 63);
  const uint16_t* a = A + (l & 15) * lda + 4 * (l >> 4);
  mlp_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kt = 0; kt < KTS; ++kt)
    if (kt < kts)
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*reinterpret_cast<const mlp_bf16x4*>(a + 16 * kt), w.b[kt], acc,
                                                      0, 0, 0);
  return acc;
}

// Forward pass and (TRAIN) backward pass to dZ1 of 16 samples per block, eight
// wavefronts: wavefront w owns hidden columns 16 w .. 16 w + 15 of both hidden
// layers -- its pre-activations stay in registers from the forward to the
// backward pass -- and output column tiles w and w + 8.  Activations pass
// between layers through LDS as BF16.  The weights were last written by other
// XCDs' compute units, so every first touch costs a trip past the L2; all of a
// wavefront's operand tiles, biases and targets are therefore loaded into
// registers up front, where one such latency covers them together (loaded
// layer by layer the kernel took 19.2 us for 512 samples of a 54-state network,
// now 15.0 us).
template <bool TRAIN>
__global__ __launch_bounds__(512) void k_mlp_rows(MlpBatch m) {
  constexpr int H = kMlpHidden, HT = H / 16, LX = 64 + kMlpPad, LH = H + kMlpPad, LY = 192 + kMlpPad;
  __shared__ __align__(16) uint16_t sx[16 * LX], sa1[16 * LH], sa2[16 * LH], sdy[16 * LY], sdz2[16 * LH];
  __shared__ double part[8];
  const int kt = blockIdx.x, KT = m.rows / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = (int)(threadIdx.x & 63);
  const int c = l & 15, r0 = 4 * (l >> 4);  // column and first row of a result register
  const int XT = m.inp / 16, YT = m.outp / 16;
  const int hc = 16 * w + c;  // hidden column of this lane
  MlpW<4> w1;
  MlpW<HT> w2, w3[2], w2t;
  MlpW<12> w3t;
  w1.load(m.w1, w, XT);
  w2.load(m.w2, w, HT);
  const float b1 = m.b1[hc], b2 = m.b2[hc];
  float b3[2] = {0.0f, 0.0f}, tg[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int nt = w + 8 * s, j = 16 * nt + c;
    if (nt >= YT) continue;
    w3[s].load(m.w3, nt, HT);
    if (j < m.out) b3[s] = m.b3[j];
    if (TRAIN) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int b = 16 * kt + r0 + i;
        const size_t row = m.idx ? m.idx[b] : b;
        tg[s][i] = j < m.out ? m.t[row * m.out + j] : 0.0f;
      }
    }
  }
  if (TRAIN) {
    w3t.load(m.w3t, w, YT);
    w2t.load(m.w2t, w, HT);
  }
  for (int e = threadIdx.x; e < 16 * m.inp; e += 512) {
    const int r = e / m.inp, j = e % m.inp, b = 16 * kt + r;
    const size_t row = m.idx ? m.idx[b] : b;
    sx[r * LX + j] = j < m.in ? mlp_bf16(m.x[row * m.in + j]) : (uint16_t)0;
  }
  __syncthreads();
  if (TRAIN && w < XT) {
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = (short)sx[(r0 + i) * LX + 16 * w + c];
    m.fx[((size_t)w * KT + kt) * 64 + l] = f;
  }
  const size_t frag = ((size_t)w * KT + kt) * 64 + l;
  float z1[4], z2[4];
  {
    const mlp_f32x4 acc = mlp_tile(sx, LX, w1, XT);
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      z1[i] = acc[i] + b1;
      f[i] = (short)mlp_bf16(mlp_gelu(z1[i]));
      sa1[(r0 + i) * LH + hc] = (uint16_t)f[i];
    }
    if (TRAIN) m.fa1[frag] = f;
  }
  __syncthreads();
  {
    const mlp_f32x4 acc = mlp_tile(sa1, LH, w2, HT);
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      z2[i] = acc[i] + b2;
      f[i] = (short)mlp_bf16(mlp_gelu(z2[i]));
      sa2[(r0 + i) * LH + hc] = (uint16_t)f[i];
    }
    if (TRAIN) m.fa2[frag] = f;
  }
  __syncthreads();
  double e2 = 0.0;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int nt = w + 8 * s;
    if (nt >= YT) continue;
    const mlp_f32x4 acc = mlp_tile(sa2, LH, w3[s], HT);
    const int j = 16 * nt + c;
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = 16 * kt + r0 + i;
      const float y = j < m.out ? acc[i] + b3[s] : 0.0f;
      if (!TRAIN) {
        if (j < m.out) m.y[(size_t)b * m.out + j] = y;
      } else {
        float d = 0.0f;
        if (j < m.out) {
          const float e = y - tg[s][i];
          d = 2.0f * e / (float)((double)m.rows * m.out);
          e2 += (double)e * e;
        }
        f[i] = (short)mlp_bf16(d);
        sdy[(r0 + i) * LY + j] = (uint16_t)f[i];
        m.dy[(size_t)b * m.outp + j] = d;
      }
    }
    if (TRAIN) m.fdy[((size_t)nt * KT + kt) * 64 + l] = f;
  }
  if (!TRAIN) return;
  // squared error of the tile, in a fixed order
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) e2 += __shfl_xor(e2, s);
  if (l == 0) part[w] = e2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int q = 0; q < 8; ++q) s += part[q];
    m.loss[kt] = s;
  }
  {
    const mlp_f32x4 acc = mlp_tile(sdy, LY, w3t, YT);
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = acc[i] * mlp_gelu_grad(z2[i]);
      f[i] = (short)mlp_bf16(d);
      sdz2[(r0 + i) * LH + hc] = (uint16_t)f[i];
      m.dz2[(size_t)(16 * kt + r0 + i) * H + hc] = d;
    }
    m.fdz2[frag] = f;
  }
  __syncthreads();
  {
    const mlp_f32x4 acc = mlp_tile(sdz2, LH, w2t, HT);
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = acc[i] * mlp_gelu_grad(z1[i]);
      f[i] = (short)mlp_bf16(d);
      m.dz1[(size_t)(16 * kt + r0 + i) * H + hc] = d;
    }
    m.fdz1[frag] = f;
  }
}

// Parameters of one Adam step (lr = 0 and adam = 0: gradients only).
struct MlpStep {
  float *p, *g, *am, *av;
  uint16_t *w1, *w2, *w3, *w2t, *w3t;  // operand tiles of the updated weights
  int off_w1, off_b1, off_w2, off_b2, off_w3, off_b3;
  int adam;
  float lr, b1, b2, eps, c1, c2;
};

// One parameter's state, loaded before its gradient is known, and its update.
struct MlpParam {
  float p, am, av;
  __device__ __forceinline__ void load(const MlpStep& s, int i) {
    p = s.p[i];
    am = s.am[i];
    av = s.av[i];
  }
  __device__ __forceinline__ float update(const MlpStep& s, int i, float gi) {
    // (fused as written: a training run repeats bit for bit across builds)
    const float mi = fmaf(1.0f - s.b1, gi, s.b1 * am);
    const float vi = fmaf(gi, (1.0f - s.b2) * gi, s.b2 * av);
    s.am[i] = mi;
    s.av[i] = vi;
    p -= s.lr * (mi / s.c1) / (sqrtf(vi / s.c2) + s.eps);
    s.p[i] = p;
    return p;
  }
};

// One wavefront per block.  Blocks 0 .. tiles - 1: a 16x16 tile of a weight
// gradient, A^T dZ over the batch from the stored fragments (row tiles in
// ascending order); the rest: 16 bias gradients, the FP32 column sums in 16 row
// phases joined in a fixed order.  Each then updates its own parameters and
// their operand tiles, so no gradient goes through memory when training.  Bound
// by latency like k_mlp_rows (12.2 us with eight fragments in flight and the
// Adam state loaded after the product, now 5.2 us).
__global__ __launch_bounds__(64) void k_mlp_weights(MlpBatch m, MlpStep s) {
  constexpr int H = kMlpHidden, HT = H / 16;
  const int l = (int)threadIdx.x, KT = m.rows / 16, XT = m.inp / 16, YT = m.outp / 16;
  int b = blockIdx.x;
  const int tiles = HT * YT + HT * HT + XT * HT;
  if (b < tiles) {
    const mlp_bf16x4 *fa, *fb;
    uint16_t *wn, *wt = nullptr;
    int off, N, mts, mt, nt;
    if (b < HT * YT) {
      fa = m.fa2, fb = m.fdy, off = s.off_w3, N = m.outp, mts = HT, mt = b / YT, nt = b % YT;
      wn = s.w3, wt = s.w3t;
    } else if (b < HT * YT + HT * HT) {
      b -= HT * YT;
      fa = m.fa1, fb = m.fdz2, off = s.off_w2, N = H, mts = HT, mt = b / HT, nt = b % HT;
      wn = s.w2, wt = s.w2t;
    } else {
      b -= HT * YT + HT * HT;
      fa = m.fx, fb = m.fdz1, off = s.off_w1, N = H, mts = XT, mt = b / HT, nt = b % HT;
      wn = s.w1;
    }
    fa += (size_t)mt * KT * 64 + l;
    fb += (size_t)nt * KT * 64 + l;
    MlpParam pr[4];
    const int at0 = off + (16 * mt + 4 * (l >> 4)) * N + 16 * nt + (l & 15);
    if (s.adam) {
#pragma unroll
      for (int i = 0; i < 4; ++i) pr[i].load(s, at0 + i * N);
    }
    mlp_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int U = 32;  // row tiles in flight (a batch of 512)
    for (int k0 = 0; k0 < KT; k0 += U) {
      mlp_bf16x4 a[U], w[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k0 + u < KT) {
          a[u] = fa[(size_t)(k0 + u) * 64];
          w[u] = fb[(size_t)(k0 + u) * 64];
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k0 + u < KT) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[u], w[u], acc, 0, 0, 0);
    }
    mlp_bf16x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 16 * mt + 4 * (l >> 4) + i, n = 16 * nt + (l & 15);
      const int at = at0 + i * N;
      if (!s.adam) {
        s.g[at] = acc[i];
        continue;
      }
      f[i] = (short)mlp_bf16(pr[i].update(s, at, acc[i]));
      // W^T[n][k] in its own operand order
      if (wt)
        wt[(((size_t)mt * (N / 16) + nt) * 64 + 16 * ((n & 15) >> 2) + (k & 15)) * 4 + (n & 3)] = (uint16_t)f[i];
    }
    if (s.adam) reinterpret_cast<mlp_bf16x4*>(wn)[((size_t)nt * mts + mt) * 64 + l] = f;
    return;
  }
  b -= tiles;
  const float* X;
  int cols, off;
  if (b < YT) {
    X = m.dy, cols = m.outp, off = s.off_b3;
  } else if (b < YT + HT) {
    b -= YT;
    X = m.dz2, cols = H, off = s.off_b2;
  } else {
    b -= YT + HT;
    X = m.dz1, cols = H, off = s.off_b1;
  }
  __shared__ float part[16][17];
  const int tx = l & 15, tq = 4 * (l >> 4), j = 16 * b + tx;
  MlpParam pr;
  if (s.adam) pr.load(s, off + j);
  float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 16
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] += X[(size_t)(16 * kt + tq + q) * cols + j];
#pragma unroll
  for (int q = 0; q < 4; ++q) part[tq + q][tx] = sum[q];
  __syncthreads();
  if (l < 16) {
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += part[k][tx];
    if (s.adam) pr.update(s, off + j, t);
    else s.g[off + j] = t;
  }
}

// FP32 K x N row-major -> BF16 in MFMA B-operand tile order (see MlpView).
__global__ void k_mlp_swizzle(int K, int N, const float* __restrict__ W, uint16_t* __restrict__ out) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= K * N) return;
  const int KT = K / 16;
  const int i = idx & 3, l = (idx >> 2) & 63, tile = idx >> 8;
  const int kt = tile % KT, nt = tile / KT;
  const int k = 16 * kt + 4 * (l >> 4) + i, n = 16 * nt + (l & 15);
  out[idx] = mlp_bf16(W[(size_t)k * N + n]);
}

// The same for the transpose of W: tiles of W^T (N x K).
__global__ void k_mlp_swizzle_t(int K, int N, const float* __restrict__ W, uint16_t* __restrict__ out) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= K * N) return;
  const int NT = N / 16;
  const int i = idx & 3, l = (idx >> 2) & 63, tile = idx >> 8;
  const int kt = tile % NT, nt = tile / NT;
  const int n = 16 * kt + 4 * (l >> 4) + i, k = 16 * nt + (l & 15);
  out[idx] = mlp_bf16(W[(size_t)k * N + n]);
}

// In-integrator inference path on given states: one wavefront per condition,
// lane r < N holding y_r (condition-major y[c*N + r]), parameter pr[c];
// z[c*3N + s*N + r].
template <int N>
__global__ __launch_bounds__(64) void k_mlp_predict_states(int num, double logh, const double* __restrict__ y,
                                                           const double* __restrict__ pr, double* __restrict__ z,
                                                           MlpView m) {
  const int c = blockIdx.x;
  if (c >= num) return;
  const int l = (int)threadIdx.x;
  const double yr = l < N ? y[(size_t)c * N + l] : 0.0;
  double z1, z2, z3;
  mlp_predict_wave<N>(m, yr, logh, log(pr[c]), z1, z2, z3);
  if (l < N) {
    z[(size_t)c * 3 * N + l] = z1;
    z[(size_t)c * 3 * N + N + l] = z2;
    z[(size_t)c * 3 * N + 2 * N + l] = z3;
  }
}

namespace {

struct Mlp {
  int n = 0;                 // system size
  int in = 0, inp = 0, out = 0, outp = 0;
  int off_w1 = 0, off_b1 = 0, off_w2 = 0, off_b2 = 0, off_w3 = 0, off_b3 = 0, count = 0;
  float* p = nullptr;        // parameters (FP32 master)
  float* g = nullptr;        // gradients
  float* am = nullptr;       // Adam moments
  float* av = nullptr;
  uint16_t* w1s = nullptr;   // BF16 swizzled copies for the integrator
  uint16_t* w2s = nullptr;
  uint16_t* w3s = nullptr;
  float* mu = nullptr;
  float* sd = nullptr;
  float* zs = nullptr;
  int adam_t = 0;
  // training's own operand tiles (the integrator keeps reading w1s, w2s, w3s):
  // one allocation at t1; fresh: they are those of p
  uint16_t *t1 = nullptr, *t2 = nullptr, *t3 = nullptr, *t2t = nullptr, *t3t = nullptr;
  bool tiles_fresh = false;
  // batch workspace (one allocation), for batches of up to cap samples
  int cap = 0;
  char* ws = nullptr;
  std::string err;
} G;

bool ok(hipError_t e, const char* what) {
  if (e == hipSuccess) return true;
  G.err = std::string(what) + ": " + hipGetErrorString(e);
  return false;
}

void free_ws() {
  if (G.ws) hipFree(G.ws);
  G.ws = nullptr;
  G.cap = 0;
}

// Bumped whenever the network's buffers are freed: a captured graph that
// reads them checks it before every replay.
int g_generation = 0;

void free_all() {
  ++g_generation;
  free_ws();
  for (float** q : {&G.p, &G.g, &G.am, &G.av, &G.mu, &G.sd, &G.zs}) {
    if (*q) hipFree(*q);
    *q = nullptr;
  }
  for (uint16_t** q : {&G.w1s, &G.w2s, &G.w3s, &G.t1}) {
    if (*q) hipFree(*q);
    *q = nullptr;
  }
  G.n = 0;
}

int blocks_for(size_t n, int t = 256) { return (int)((n + t - 1) / t); }

// The batch's buffers in the workspace (base 0: their total size in `bytes`).
MlpBatch batch_buffers(int B, char* base, size_t* bytes) {
  const size_t H = kMlpHidden;
  size_t at = 0;
  auto take = [&](size_t n) {
    char* p = base + at;
    at += (n + 255) / 256 * 256;
    return p;
  };
  MlpBatch m{};
  m.in = G.in;
  m.inp = G.inp;
  m.out = G.out;
  m.outp = G.outp;
  m.rows = B;
  m.w1 = G.t1;
  m.w2 = G.t2;
  m.w3 = G.t3;
  m.w2t = G.t2t;
  m.w3t = G.t3t;
  m.b1 = G.p + G.off_b1;
  m.b2 = G.p + G.off_b2;
  m.b3 = G.p + G.off_b3;
  m.fx = (mlp_bf16x4*)take((size_t)B * G.inp * 2);
  m.fa1 = (mlp_bf16x4*)take((size_t)B * H * 2);
  m.fa2 = (mlp_bf16x4*)take((size_t)B * H * 2);
  m.fdy = (mlp_bf16x4*)take((size_t)B * G.outp * 2);
  m.fdz2 = (mlp_bf16x4*)take((size_t)B * H * 2);
  m.fdz1 = (mlp_bf16x4*)take((size_t)B * H * 2);
  m.dy = (float*)take((size_t)B * G.outp * 4);
  m.dz2 = (float*)take((size_t)B * H * 4);
  m.dz1 = (float*)take((size_t)B * H * 4);
  // host-array calls: the uploaded samples and targets, the outputs
  m.x = (float*)take((size_t)B * G.in * 4);
  m.t = (float*)take((size_t)B * G.out * 4);
  m.y = (float*)take((size_t)B * G.out * 4);
  m.loss = (double*)take((size_t)(B / 16) * sizeof(double));
  *bytes = at;
  return m;
}

bool ensure_ws(int B) {
  if (B <= G.cap) return true;
  free_ws();
  size_t bytes = 0;
  batch_buffers(B, nullptr, &bytes);
  if (!ok(hipMalloc(&G.ws, bytes), "hipMalloc")) return false;
  G.cap = B;
  return true;
}
MlpBatch workspace_batch(int B) {
  size_t bytes = 0;
  return batch_buffers(B, G.ws, &bytes);
}

MlpStep step_params(int adam, float lr, float c1, float c2) {
  MlpStep s{};
  s.p = G.p;
  s.g = G.g;
  s.am = G.am;
  s.av = G.av;
  s.w1 = G.t1;
  s.w2 = G.t2;
  s.w3 = G.t3;
  s.w2t = G.t2t;
  s.w3t = G.t3t;
  s.off_w1 = G.off_w1;
  s.off_b1 = G.off_b1;
  s.off_w2 = G.off_w2;
  s.off_b2 = G.off_b2;
  s.off_w3 = G.off_w3;
  s.off_b3 = G.off_b3;
  s.adam = adam;
  s.lr = lr;
  s.b1 = 0.9f;
  s.b2 = 0.999f;
  s.eps = 1e-8f;
  s.c1 = c1;
  s.c2 = c2;
  return s;
}

// Squared error and gradients of a batch; with an Adam step, the parameters'
// update in place of the gradients.
void launch_batch(const MlpBatch& m, const MlpStep& s) {
  const int HT = kMlpHidden / 16, XT = m.inp / 16, YT = m.outp / 16;
  hipLaunchKernelGGL(k_mlp_rows<true>, dim3(m.rows / 16), dim3(512), 0, 0, m);
  hipLaunchKernelGGL(k_mlp_weights, dim3(HT * YT + HT * HT + XT * HT + YT + 2 * HT), dim3(64), 0, 0, m, s);
}

// Training's operand tiles from the FP32 parameters (an Adam step keeps them).
bool refresh_training_tiles() {
  if (G.tiles_fresh) return true;
  const int H = kMlpHidden;
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)G.inp * H)), dim3(256), 0, 0, G.inp, H, G.p + G.off_w1, G.t1);
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)H * H)), dim3(256), 0, 0, H, H, G.p + G.off_w2, G.t2);
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)H * G.outp)), dim3(256), 0, 0, H, G.outp, G.p + G.off_w3,
                     G.t3);
  hipLaunchKernelGGL(k_mlp_swizzle_t, dim3(blocks_for((size_t)H * H)), dim3(256), 0, 0, H, H, G.p + G.off_w2, G.t2t);
  hipLaunchKernelGGL(k_mlp_swizzle_t, dim3(blocks_for((size_t)H * G.outp)), dim3(256), 0, 0, H, G.outp,
                     G.p + G.off_w3, G.t3t);
  G.tiles_fresh = ok(hipGetLastError(), "mlp swizzle");
  return G.tiles_fresh;
}

bool refresh_swizzled() {
  const int H = kMlpHidden;
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)G.inp * H)), dim3(256), 0, 0, G.inp, H, G.p + G.off_w1,
                     G.w1s);
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)H * H)), dim3(256), 0, 0, H, H, G.p + G.off_w2, G.w2s);
  hipLaunchKernelGGL(k_mlp_swizzle, dim3(blocks_for((size_t)H * G.outp)), dim3(256), 0, 0, H, G.outp,
                     G.p + G.off_w3, G.w3s);
  return ok(hipGetLastError(), "mlp swizzle") && ok(hipDeviceSynchronize(), "mlp swizzle");
}

}  // namespace

int mlp_generation() { return g_generation; }

MlpView mlp_view() {
  MlpView v{};
  if (G.n == 0) return v;
  v.w1 = G.w1s;
  v.w2 = G.w2s;
  v.w3 = G.w3s;
  v.b1 = G.p + G.off_b1;
  v.b2 = G.p + G.off_b2;
  v.b3 = G.p + G.off_b3;
  v.mu = G.mu;
  v.sd = G.sd;
  v.zs = G.zs;
  v.n = G.n;
  v.on = 1;
  return v;
}

}  // namespace acc

using namespace acc;

extern "C" {

int accelerInt_mlp_init(int n_states, unsigned seed) {
  if (n_states < 1 || n_states + 2 > 64) {
    G.err = "accelerInt_mlp_init: n_states must be in 1..62";
    return -1;
  }
  free_all();
  const int H = kMlpHidden;
  G.n = n_states;
  G.in = n_states + 2;
  G.inp = mlp_pad16(G.in);
  G.out = 3 * n_states;
  G.outp = mlp_pad16(G.out);
  G.off_w1 = 0;
  G.off_b1 = G.off_w1 + G.inp * H;
  G.off_w2 = G.off_b1 + H;
  G.off_b2 = G.off_w2 + H * H;
  G.off_w3 = G.off_b2 + H;
  G.off_b3 = G.off_w3 + H * G.outp;
  G.count = G.off_b3 + G.outp;
  // Glorot-uniform weights over the valid rows/columns, zero padding and biases
  std::vector<float> p(G.count, 0.0f);
  std::mt19937 rng(seed);
  auto fill = [&](int off, int K, int N, int kv, int nv) {
    const float a = sqrtf(6.0f / (float)(kv + nv));
    std::uniform_real_distribution<float> u(-a, a);
    for (int k = 0; k < K; ++k)
      for (int n = 0; n < N; ++n) p[off + k * N + n] = (k < kv && n < nv) ? u(rng) : 0.0f;
  };
  fill(G.off_w1, G.inp, H, G.in, H);
  fill(G.off_w2, H, H, H, H);
  fill(G.off_w3, H, G.outp, H, G.out);
  std::vector<float> one(G.outp > G.inp ? G.outp : G.inp, 1.0f), zero(G.inp, 0.0f);
  bool good = ok(hipMalloc(&G.p, G.count * 4), "hipMalloc") && ok(hipMalloc(&G.g, G.count * 4), "hipMalloc") &&
              ok(hipMalloc(&G.am, G.count * 4), "hipMalloc") && ok(hipMalloc(&G.av, G.count * 4), "hipMalloc") &&
              ok(hipMalloc(&G.w1s, (size_t)G.inp * H * 2), "hipMalloc") &&
              ok(hipMalloc(&G.w2s, (size_t)H * H * 2), "hipMalloc") &&
              ok(hipMalloc(&G.w3s, (size_t)H * G.outp * 2), "hipMalloc") &&
              ok(hipMalloc(&G.t1, ((size_t)G.inp * H + 2 * (size_t)H * H + 2 * (size_t)H * G.outp) * 2), "hipMalloc") &&
              ok(hipMalloc(&G.mu, G.inp * 4), "hipMalloc") && ok(hipMalloc(&G.sd, G.inp * 4), "hipMalloc") &&
              ok(hipMalloc(&G.zs, G.outp * 4), "hipMalloc") &&
              ok(hipMemcpy(G.p, p.data(), G.count * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
              ok(hipMemset(G.am, 0, G.count * 4), "hipMemset") && ok(hipMemset(G.av, 0, G.count * 4), "hipMemset") &&
              ok(hipMemset(G.g, 0, G.count * 4), "hipMemset") &&
              ok(hipMemcpy(G.mu, zero.data(), G.inp * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
              ok(hipMemcpy(G.sd, one.data(), G.inp * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
              ok(hipMemcpy(G.zs, one.data(), G.outp * 4, hipMemcpyHostToDevice), "hipMemcpy") && refresh_swizzled();
  if (!good) {
    free_all();
    return -1;
  }
  G.t2 = G.t1 + (size_t)G.inp * H;
  G.t2t = G.t2 + (size_t)H * H;
  G.t3 = G.t2t + (size_t)H * H;
  G.t3t = G.t3 + (size_t)H * G.outp;
  G.tiles_fresh = false;
  G.adam_t = 0;
  return 0;
}

int accelerInt_mlp_param_count(void) { return G.n ? G.count : -1; }

int accelerInt_mlp_get_params(float* out, int count) {
  if (!G.n || count != G.count || !out) {
    G.err = "accelerInt_mlp_get_params: no network or wrong count";
    return -1;
  }
  return ok(hipMemcpy(out, G.p, (size_t)count * 4, hipMemcpyDeviceToHost), "hipMemcpy") ? 0 : -1;
}

int accelerInt_mlp_set_params(const float* in, int count) {
  if (!G.n || count != G.count || !in) {
    G.err = "accelerInt_mlp_set_params: no network or wrong count";
    return -1;
  }
  G.tiles_fresh = false;
  if (!ok(hipMemcpy(G.p, in, (size_t)count * 4, hipMemcpyHostToDevice), "hipMemcpy")) return -1;
  return refresh_swizzled() ? 0 : -1;
}

int accelerInt_mlp_set_normalization(const float* mu, const float* sd, const float* zscale) {
  if (!G.n || !mu || !sd || !zscale) {
    G.err = "accelerInt_mlp_set_normalization: no network or null array";
    return -1;
  }
  std::vector<float> m(G.inp, 0.0f), s(G.inp, 1.0f), z(G.outp, 0.0f);
  for (int j = 0; j < G.in; ++j) {
    if (!(sd[j] > 0.0f)) {
      G.err = "accelerInt_mlp_set_normalization: scales must be positive";
      return -1;
    }
    m[j] = mu[j];
    s[j] = sd[j];
  }
  for (int j = 0; j < G.out; ++j) z[j] = zscale[j];
  return ok(hipMemcpy(G.mu, m.data(), G.inp * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
                 ok(hipMemcpy(G.sd, s.data(), G.inp * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
                 ok(hipMemcpy(G.zs, z.data(), G.outp * 4, hipMemcpyHostToDevice), "hipMemcpy")
             ? 0
             : -1;
}

int accelerInt_mlp_loss_grad(int B, const float* x, const float* t, float* grad, float* loss) {
  if (!G.n || B <= 0 || B % 16 || !x || !t || !grad) {
    G.err = "accelerInt_mlp_loss_grad: no network, or B not a positive multiple of 16";
    return -1;
  }
  if (!ensure_ws(B)) return -1;
  const MlpBatch m = workspace_batch(B);
  if (!ok(hipMemcpy((void*)m.x, x, (size_t)B * G.in * 4, hipMemcpyHostToDevice), "hipMemcpy") ||
      !ok(hipMemcpy((void*)m.t, t, (size_t)B * G.out * 4, hipMemcpyHostToDevice), "hipMemcpy") ||
      !refresh_training_tiles())
    return -1;
  launch_batch(m, step_params(0, 0.0f, 1.0f, 1.0f));
  if (!ok(hipGetLastError(), "mlp backward")) return -1;
  std::vector<double> part(B / 16);
  if (!ok(hipMemcpy(part.data(), m.loss, part.size() * sizeof(double), hipMemcpyDeviceToHost), "hipMemcpy")) return -1;
  double sse = 0.0;
  for (double v : part) sse += v;
  if (loss) *loss = (float)(sse / ((double)B * G.out));
  return ok(hipMemcpy(grad, G.g, (size_t)G.count * 4, hipMemcpyDeviceToHost), "hipMemcpy") ? 0 : -1;
}

int accelerInt_mlp_predict(int B, const float* x, float* y) {
  if (!G.n || B <= 0 || B % 16 || !x || !y) {
    G.err = "accelerInt_mlp_predict: no network, or B not a positive multiple of 16";
    return -1;
  }
  if (!ensure_ws(B)) return -1;
  const MlpBatch m = workspace_batch(B);
  if (!ok(hipMemcpy((void*)m.x, x, (size_t)B * G.in * 4, hipMemcpyHostToDevice), "hipMemcpy") ||
      !refresh_training_tiles())
    return -1;
  hipLaunchKernelGGL(k_mlp_rows<false>, dim3(B / 16), dim3(512), 0, 0, m);
  return ok(hipGetLastError(), "mlp forward") &&
                 ok(hipMemcpy(y, m.y, (size_t)B * G.out * 4, hipMemcpyDeviceToHost), "hipMemcpy")
             ? 0
             : -1;
}

// Adam over shuffled batches.  An epoch's batches are launched without waiting
// for any of them; the next epoch's permutation is drawn while they run, and the
// epoch's squared errors come back in one copy at its end.
int accelerInt_mlp_train(int n, const float* x_dev, const float* t_dev, int epochs, int batch, float lr,
                         unsigned seed, float* loss_per_epoch) {
  if (!G.n || n < batch || batch <= 0 || batch % 16 || epochs <= 0 || !x_dev || !t_dev) {
    G.err = "accelerInt_mlp_train: bad arguments (batch a multiple of 16, n >= batch)";
    return -1;
  }
  if (!ensure_ws(batch)) return -1;
  std::mt19937 rng(seed);
  std::vector<int> perm(n);
  for (int i = 0; i < n; ++i) perm[i] = i;
  const int steps = n / batch, tiles = batch / 16;
  std::vector<double> part((size_t)steps * tiles);
  int* d_perm = nullptr;
  double* d_loss = nullptr;
  int rc = -1;
  if (ok(hipMalloc(&d_perm, (size_t)n * sizeof(int)), "hipMalloc") &&
      ok(hipMalloc(&d_loss, part.size() * sizeof(double)), "hipMalloc") && refresh_training_tiles())
    rc = 0;
  MlpBatch m = workspace_batch(batch);
  m.x = x_dev;
  m.t = t_dev;
  if (rc == 0) std::shuffle(perm.begin(), perm.end(), rng);
  for (int ep = 0; ep < epochs && rc == 0; ++ep) {
    if (!ok(hipMemcpy(d_perm, perm.data(), (size_t)n * sizeof(int), hipMemcpyHostToDevice), "hipMemcpy")) {
      rc = -1;
      break;
    }
    for (int s = 0; s < steps; ++s) {
      m.idx = d_perm + (size_t)s * batch;
      m.loss = d_loss + (size_t)s * tiles;
      ++G.adam_t;
      const float c1 = 1.0f - powf(0.9f, (float)G.adam_t), c2 = 1.0f - powf(0.999f, (float)G.adam_t);
      launch_batch(m, step_params(1, lr, c1, c2));
    }
    if (!ok(hipGetLastError(), "mlp training")) {
      rc = -1;
      break;
    }
    if (ep + 1 < epochs) std::shuffle(perm.begin(), perm.end(), rng);
    if (!ok(hipMemcpy(part.data(), d_loss, part.size() * sizeof(double), hipMemcpyDeviceToHost), "hipMemcpy")) {
      rc = -1;
      break;
    }
    double sse = 0.0;
    for (double v : part) sse += v;
    if (loss_per_epoch) loss_per_epoch[ep] = (float)(sse / ((double)steps * batch * G.out));
    if (!std::isfinite(sse)) {
      G.err = "accelerInt_mlp_train: non-finite loss (training diverged or non-finite samples)";
      rc = -1;
    }
  }
  if (d_perm) hipFree(d_perm);
  if (d_loss) hipFree(d_loss);
  if (rc == 0 && !refresh_swizzled()) rc = -1;
  return rc;
}

int accelerInt_mlp_predict_states(int num, double h, const double* y, const double* pr, double* z) {
  if (G.n != 54 || num <= 0 || !y || !pr || !z || !(h > 0)) {
    G.err = "accelerInt_mlp_predict_states: needs a 54-state network, num > 0, h > 0";
    return -1;
  }
  const int N = 54;
  double *dy = nullptr, *dz = nullptr, *dp = nullptr;
  int rc = -1;
  if (ok(hipMalloc(&dy, (size_t)num * N * 8), "hipMalloc") && ok(hipMalloc(&dz, (size_t)num * 3 * N * 8), "hipMalloc") &&
      ok(hipMalloc(&dp, (size_t)num * 8), "hipMalloc") &&
      ok(hipMemcpy(dy, y, (size_t)num * N * 8, hipMemcpyHostToDevice), "hipMemcpy") &&
      ok(hipMemcpy(dp, pr, (size_t)num * 8, hipMemcpyHostToDevice), "hipMemcpy")) {
    hipLaunchKernelGGL(k_mlp_predict_states<54>, dim3(num), dim3(64), 0, 0, num, log(h), dy, dp, dz, mlp_view());
    if (ok(hipGetLastError(), "k_mlp_predict_states") &&
        ok(hipMemcpy(z, dz, (size_t)num * 3 * N * 8, hipMemcpyDeviceToHost), "hipMemcpy"))
      rc = 0;
  }
  if (dy) hipFree(dy);
  if (dz) hipFree(dz);
  if (dp) hipFree(dp);
  return rc;
}

int accelerInt_mlp_train_host(int n, const float* x, const float* t, int epochs, int batch, float lr, unsigned seed,
                              float* loss_per_epoch) {
  if (!G.n || n <= 0 || !x || !t) {
    G.err = "accelerInt_mlp_train_host: no network or empty data";
    return -1;
  }
  float *dx = nullptr, *dt = nullptr;
  int rc = -1;
  if (ok(hipMalloc(&dx, (size_t)n * G.in * 4), "hipMalloc") && ok(hipMalloc(&dt, (size_t)n * G.out * 4), "hipMalloc") &&
      ok(hipMemcpy(dx, x, (size_t)n * G.in * 4, hipMemcpyHostToDevice), "hipMemcpy") &&
      ok(hipMemcpy(dt, t, (size_t)n * G.out * 4, hipMemcpyHostToDevice), "hipMemcpy"))
    rc = accelerInt_mlp_train(n, dx, dt, epochs, batch, lr, seed, loss_per_epoch);
  if (dx) hipFree(dx);
  if (dt) hipFree(dt);
  return rc;
}

const char* accelerInt_mlp_last_error(void) { return G.err.c_str(); }

void accelerInt_mlp_release(void) { free_all(); }

}  // extern "C"
