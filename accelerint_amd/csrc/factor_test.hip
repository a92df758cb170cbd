// Device LU without integration: the LU routines the integrator runs at each
// order and precision (radau_core.hpp: the row LU lu_real / lu_cplx with
// implicit interchanges; at order 14 row16_lu_real / row16_lu_cplx, which leave
// the rows in LAPACK's order) on caller matrices, so that their pivot
// choice, factors and zero-pivot report can be checked one to one against
// LAPACK dgetrf_/zgetrf_, the routines the reference calls in RK_Decomp
// (radau2a.c:273,277); optionally also the matching triangular solves on one
// right-hand side per matrix, the counterpart of dgetrs_ / zgetrs_
// (radau2a.c:404,417).  Orders 2 (one system per lane), 14 (16-lane
// groups), 54 (one wave per system) and 112 (one wave per system, the
// memory-resident blocked LU with MFMA trailing updates).
#include <hip/hip_runtime.h>

#include "radau_core.hpp"

namespace acc {

// One group per matrix.  a_re/a_im: row-major N x N per matrix (a_im unused
// for the real LU).  Row r of the factored matrix is written to the row of
// the LAPACK factors it ends at (its elimination step pos), so lu holds the
// combined unit-L / U factors of P A as dgetrf_ returns them; perm[k] = the
// original row chosen as pivot at step k; info as dgetrf_.  With b_re set,
// x = A^-1 b from the factors (b_im / x_im: imaginary parts, complex LU).
template <int N, int G, int R, class T, bool CPLX>
__global__ __launch_bounds__(64) void k_factor_test(int num, const double* __restrict__ a_re,
                                                    const double* __restrict__ a_im, const double* __restrict__ b_re,
                                                    const double* __restrict__ b_im, double* __restrict__ lu_re,
                                                    double* __restrict__ lu_im, int* __restrict__ perm_out,
                                                    int* __restrict__ info_out, double* __restrict__ x_re,
                                                    double* __restrict__ x_im) {
  using RW = Rows<N, G, R>;
  const int ln = Grp<G>::lane();
  const int c = blockIdx.x * (64 / G) + (int)threadIdx.x / G;
  if (c >= num) return;  // whole groups leave together
  const size_t base = (size_t)c * N * N;
  T ar[R][N], ai[R][N];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool v = RW::valid(ln, q);
    const int r = RW::row(ln, q);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      ar[q][j] = v ? (T)a_re[base + (size_t)r * N + j] : T(0);
      ai[q][j] = (CPLX && v) ? (T)a_im[base + (size_t)r * N + j] : T(0);
    }
  }
  int pos[R];
  Perm<N> perm;
#pragma unroll
  for (int i = 0; i < (N + 3) / 4; ++i) perm.w[i] = 0;
  T rdr[R], rdi[R];
  int info = 0;
  if constexpr (G == 64 && R == 1) {
    // the other factorization of the pair works on the same real parts
    T br[R][N], bi[R][N], d[R], di[R];
    int p2[R], inf2;
    Perm<N> q;
#pragma unroll
    for (int j = 0; j < N; ++j) br[0][j] = ar[0][j], bi[0][j] = ai[0][j];
    if constexpr (CPLX) wave_lu<N, T>(br, p2, q, d, inf2, ar, ai, pos, perm, rdr, rdi, info);
    else wave_lu<N, T>(ar, pos, perm, rdr, info, br, bi, p2, q, d, di, inf2);
  } else if constexpr (CPLX) lu_cplx<N, G, R, T>(ar, ai, pos, perm, rdr, rdi, info);
  else lu_real<N, G, R, T>(ar, pos, perm, rdr, info);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    if (RW::valid(ln, q) && pos[q] >= 0 && pos[q] < N) {
      const size_t o = base + (size_t)pos[q] * N;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        lu_re[o + j] = (double)ar[q][j];
        if (CPLX) lu_im[o + j] = (double)ai[q][j];
      }
    }
  }
  if (ln == 0) {
    for (int k = 0; k < N; ++k) perm_out[(size_t)c * N + k] = perm.get(k);
    info_out[c] = info;
  }
  if (b_re) {  // uniform over the launch
    T br[R], bi[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const bool v = RW::valid(ln, q);
      const size_t o = (size_t)c * N + RW::row(ln, q);
      br[q] = v ? (T)b_re[o] : T(0);
      bi[q] = (CPLX && v) ? (T)b_im[o] : T(0);
    }
    if constexpr (CPLX) solve_cplx<N, G, R, T>(ar, ai, pos, perm, rdr, rdi, br, bi);
    else solve_real<N, G, R, T>(ar, pos, perm, rdr, br);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (RW::valid(ln, q)) {
        const size_t o = (size_t)c * N + RW::row(ln, q);
        x_re[o] = (double)br[q];
        if (CPLX) x_im[o] = (double)bi[q];
      }
    }
  }
}

// Order 14: the LU of 16-lane groups, rows moved to the lanes of their LAPACK
// positions (src = the original row now in this lane, which is also the row
// chosen at that step), and its solves.
template <class T, bool CPLX>
__global__ __launch_bounds__(64) void k_factor_test_16(int num, const double* __restrict__ a_re,
                                                       const double* __restrict__ a_im,
                                                       const double* __restrict__ b_re,
                                                       const double* __restrict__ b_im, double* __restrict__ lu_re,
                                                       double* __restrict__ lu_im, int* __restrict__ perm_out,
                                                       int* __restrict__ info_out, double* __restrict__ x_re,
                                                       double* __restrict__ x_im) {
  constexpr int N = 14, G = 16;
  const int ln = Grp<G>::lane();
  const int c = blockIdx.x * (64 / G) + (int)threadIdx.x / G;
  if (c >= num) return;  // whole groups leave together
  const size_t base = (size_t)c * N * N;
  T ar[N], ai[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    ar[j] = ln < N ? (T)a_re[base + (size_t)ln * N + j] : T(0);
    ai[j] = (CPLX && ln < N) ? (T)a_im[base + (size_t)ln * N + j] : T(0);
  }
  int src = 0, info = 0;
  T rdr, rdi = T(0);
  if constexpr (CPLX) row16_lu_cplx<N, T>(ar, ai, src, rdr, rdi, info);
  else row16_lu_real<N, T>(ar, src, rdr, info);
  if (ln < N) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      lu_re[base + (size_t)ln * N + j] = (double)ar[j];
      if (CPLX) lu_im[base + (size_t)ln * N + j] = (double)ai[j];
    }
    perm_out[(size_t)c * N + ln] = src;
  }
  if (ln == 0) info_out[c] = info;
  if (b_re) {  // uniform over the launch
    T br = ln < N ? (T)b_re[(size_t)c * N + ln] : T(0);
    T bi = (CPLX && ln < N) ? (T)b_im[(size_t)c * N + ln] : T(0);
    if constexpr (CPLX) rsolve_cplx<N, G, T>(ar, ai, src, rdr, rdi, br, bi);
    else rsolve_real<N, G, T>(ar, src, rdr, br);
    if (ln < N) {
      x_re[(size_t)c * N + ln] = (double)br;
      if (CPLX) x_im[(size_t)c * N + ln] = (double)bi;
    }
  }
}

// Order 112: the memory-resident blocked LU of the large systems (MemLU, one
// wave per matrix, factors in the workspace ws: MemLU<112, 2, double>::bytes()
// per matrix); perm[k] = the original row that ends at position k (the row
// chosen at step k).
template <class T, bool CPLX>
__global__ __launch_bounds__(64) void k_factor_test_mem(int num, const double* __restrict__ a_re,
                                                        const double* __restrict__ a_im,
                                                        const double* __restrict__ b_re,
                                                        const double* __restrict__ b_im, double* __restrict__ lu_re,
                                                        double* __restrict__ lu_im, int* __restrict__ perm_out,
                                                        int* __restrict__ info_out, double* __restrict__ x_re,
                                                        double* __restrict__ x_im, char* __restrict__ ws) {
  constexpr int N = 112, R = 2;
  using MLU = MemLU<N, R, T>;
  constexpr int LD = MLU::LD;
  const int c = blockIdx.x;
  if (c >= num) return;
  const int ln = (int)threadIdx.x;
  T* E1 = reinterpret_cast<T*>(ws + (size_t)c * MemLU<N, R, double>::bytes());
  T* E2r = E1 + MLU::kMat;
  T* E2i = E2r + MLU::kMat;
  int* perm = CPLX ? MLU::perm2(E1) : MLU::perm1(E1);
  T* Er = CPLX ? E2r : E1;
  const size_t base = (size_t)c * N * N;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = ln + 64 * q;
    if (r < N) {
      for (int j = 0; j < N; ++j) {
        Er[(size_t)j * LD + r] = (T)a_re[base + (size_t)r * N + j];
        if (CPLX) E2i[(size_t)j * LD + r] = (T)a_im[base + (size_t)r * N + j];
      }
    }
  }
  wave_vmem_sync();
  int info = 0;
  if constexpr (CPLX) MLU::factor_cplx(E2r, E2i, perm, MLU::tmp(E1), info);
  else MLU::factor_real(E1, perm, MLU::tmp(E1), info);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = ln + 64 * q;
    if (r < N) {
      for (int j = 0; j < N; ++j) {
        lu_re[base + (size_t)r * N + j] = (double)Er[(size_t)j * LD + r];
        if (CPLX) lu_im[base + (size_t)r * N + j] = (double)E2i[(size_t)j * LD + r];
      }
    }
  }
  if (ln == 0) {
    for (int k = 0; k < N; ++k) perm_out[(size_t)c * N + k] = perm[k];
    info_out[c] = info;
  }
  if (b_re) {  // uniform over the launch
    T br[R], bi[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + 64 * q;
      br[q] = r < N ? (T)b_re[(size_t)c * N + r] : T(0);
      bi[q] = (CPLX && r < N) ? (T)b_im[(size_t)c * N + r] : T(0);
    }
    if constexpr (CPLX) MLU::solve_cplx(E2r, E2i, perm, br, bi);
    else MLU::solve_real(E1, perm, br);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + 64 * q;
      if (r < N) {
        x_re[(size_t)c * N + r] = (double)br[q];
        if (CPLX) x_im[(size_t)c * N + r] = (double)bi[q];
      }
    }
  }
}

template <int N, int G, int R, class T, bool CPLX>
static hipError_t launch_one(int num, const double* are, const double* aim, const double* bre, const double* bim,
                             double* lre, double* lim, int* perm, int* info, double* xre, double* xim,
                             hipStream_t s) {
  constexpr int per_block = 64 / G;
  const int blocks = (num + per_block - 1) / per_block;
  hipLaunchKernelGGL((k_factor_test<N, G, R, T, CPLX>), dim3(blocks), dim3(64), 0, s, num, are, aim, bre, bim, lre,
                     lim, perm, info, xre, xim);
  return hipGetLastError();
}

template <int N, int G, int R>
static hipError_t launch_order(bool fp32, bool cplx, int num, const double* are, const double* aim,
                               const double* bre, const double* bim, double* lre, double* lim, int* perm, int* info,
                               double* xre, double* xim, hipStream_t s) {
  if (fp32) {
    return cplx ? launch_one<N, G, R, float, true>(num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s)
                : launch_one<N, G, R, float, false>(num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s);
  }
  return cplx ? launch_one<N, G, R, double, true>(num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s)
              : launch_one<N, G, R, double, false>(num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s);
}

// Device buffers of num matrices of order n (2, 14, 54 or 112; for 112 also
// the workspace ws of num * factor_test_ws_bytes(112)); bre = nullptr: no
// solve.  Returns hipErrorInvalidValue for any other order.
size_t factor_test_ws_bytes(int n) { return n == 112 ? MemLU<112, 2, double>::bytes() : 0; }

hipError_t launch_factor_test(int n, bool fp32, bool cplx, int num, const double* are, const double* aim,
                              const double* bre, const double* bim, double* lre, double* lim, int* perm, int* info,
                              double* xre, double* xim, char* ws, hipStream_t s) {
  if (n == 112) {
    if (!ws) return hipErrorInvalidValue;
    if (fp32) {
      if (cplx)
        hipLaunchKernelGGL((k_factor_test_mem<float, true>), dim3(num), dim3(64), 0, s, num, are, aim, bre, bim, lre,
                           lim, perm, info, xre, xim, ws);
      else
        hipLaunchKernelGGL((k_factor_test_mem<float, false>), dim3(num), dim3(64), 0, s, num, are, aim, bre, bim, lre,
                           lim, perm, info, xre, xim, ws);
    } else {
      if (cplx)
        hipLaunchKernelGGL((k_factor_test_mem<double, true>), dim3(num), dim3(64), 0, s, num, are, aim, bre, bim, lre,
                           lim, perm, info, xre, xim, ws);
      else
        hipLaunchKernelGGL((k_factor_test_mem<double, false>), dim3(num), dim3(64), 0, s, num, are, aim, bre, bim,
                           lre, lim, perm, info, xre, xim, ws);
    }
    return hipGetLastError();
  }
  switch (n) {
    case 2: return launch_order<2, 1, 2>(fp32, cplx, num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s);
    case 14: {
      const dim3 blocks((num + 3) / 4);
#define LAUNCH_16(T, CPLX)                                                                                       \
  hipLaunchKernelGGL((k_factor_test_16<T, CPLX>), blocks, dim3(64), 0, s, num, are, aim, bre, bim, lre, lim, perm, \
                     info, xre, xim)
      if (fp32 && cplx) LAUNCH_16(float, true);
      else if (fp32) LAUNCH_16(float, false);
      else if (cplx) LAUNCH_16(double, true);
      else LAUNCH_16(double, false);
#undef LAUNCH_16
      return hipGetLastError();
    }
    case 54: return launch_order<54, 64, 1>(fp32, cplx, num, are, aim, bre, bim, lre, lim, perm, info, xre, xim, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace acc
