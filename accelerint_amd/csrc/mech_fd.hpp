// Finite-difference Jacobian over any mechanism's dydt: the reference's
// generic/fd_jacob.c:24-127 for FD_ORD 1 (its default), 2, 4 and 6, for
// callbacks that come without an analytic Jacobian.  Per column j, with
// ewt_i = atol + rtol |y_i| (the tolerances themselves, as the reference uses
// them):
//   fac = sqrt(sum_i (ewt_i f_i)^2 / N),  r0 = 1000 rtol eps N fac,
//   r   = max(sqrt(eps) |y_j|, r0 / ewt_j),
//   order 1:    J(:, j) = (f(y + r e_j) - f(y)) / r,
//   order 2m:   J(:, j) = (sum_k w_k f(y + x_k r e_j)) / r over the central
//               stencil of order 2m (fd_stencil below), summed in k order.
// Order 1 takes N + 1 dydt evaluations per Jacobian, order p takes p N + 1.
// Each lane writes the entries of the rows it owns, into the same place the
// base mechanism's analytic Jacobian goes (registers, or the group's LDS rows).
#pragma once

#include <float.h>

#include "radau_core.hpp"

namespace acc {

// Central-difference stencils of orders 2, 4 and 6: offsets x_k (in units of
// the increment r) and weights w_k, the textbook values that make
// sum_k w_k f(x_k r) / r exact for polynomials of degree <= order (weights
// antisymmetric, sum_k w_k x_k = 1, higher moments zero up to the order).
__host__ __device__ inline void fd_stencil(int order, int k, double& x, double& w) {
  switch (order) {
    case 2: {
      x = k == 0 ? -1.0 : 1.0;
      w = k == 0 ? -0.5 : 0.5;
      break;
    }
    case 4: {
      const double xs[4] = {-2.0, -1.0, 1.0, 2.0};
      const double ws[4] = {1.0 / 12.0, -2.0 / 3.0, 2.0 / 3.0, -1.0 / 12.0};
      x = xs[k];
      w = ws[k];
      break;
    }
    default: {  // 6
      const double xs[6] = {-3.0, -2.0, -1.0, 1.0, 2.0, 3.0};
      const double ws[6] = {-1.0 / 60.0, 3.0 / 20.0, -3.0 / 4.0, 3.0 / 4.0, -3.0 / 20.0, 1.0 / 60.0};
      x = xs[k];
      w = ws[k];
      break;
    }
  }
}

template <class Base>
struct MechFD {
  static constexpr int N = Base::N;
  static constexpr bool kJacInLds = Base::kJacInLds;
  static constexpr bool kJacColMajor = JacColMajor<Base>::value;
  static constexpr int kJacLd = JacLd<Base>::value;
  struct Params {
    typename Base::Params base;
    double atol, rtol;
    int order;  // 1, 2, 4 or 6
  };
  static size_t lds_bytes(const Params& p, int groups) {
    return Base::lds_bytes(p.base, groups);
  }
  __device__ __forceinline__ static void block_init(const Params& p, double* lds) { Base::block_init(p.base, lds); }
  struct Ctx : Base::Ctx {
    double atol, rtol;
    int order;
    __device__ Ctx(const Params& p, int g, double* lds)
        : Base::Ctx(p.base, g, lds), atol(p.atol), rtol(p.rtol), order(p.order) {}
    __device__ Ctx(const Params& p, const double* tables, double* group)
        : Base::Ctx(p.base, tables, group), atol(p.atol), rtol(p.rtol), order(p.order) {}
  };

  template <int G, int R>
  __device__ __forceinline__ static void dydt(Ctx& c, double t, double pr, const double (&y)[R], double (&f)[R]) {
    Base::template dydt<G, R>(c, t, pr, y, f);
  }

  // Column j of the difference quotient, passed to put(j, col) (col[q] = the
  // entry of row ln + G q).
  template <int G, int R, class Put>
  __device__ __forceinline__ static void columns(Ctx& c, double t, double pr, const double (&y)[R], Put&& put) {
    using RW = Rows<N, G, R>;
    const int ln = Grp<G>::lane();
    double f0[R];
    Base::template dydt<G, R>(c, t, pr, y, f0);
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double ew = c.atol + c.rtol * fabs(y[q]);
      if (RW::valid(ln, q)) s += (ew * f0[q]) * (ew * f0[q]);
    }
    s = Grp<G>::sum(s);
    const double fac = sqrt(s / (double)N);
    const double r0 = 1000.0 * c.rtol * DBL_EPSILON * (double)N * fac;
    const double srur = sqrt(DBL_EPSILON);
#pragma unroll 1
    for (int j = 0; j < N; ++j) {
      double mine[R];
#pragma unroll
      for (int q = 0; q < R; ++q) mine[q] = y[q];
      const double yj = Grp<G>::bcast(sel<R>(mine, j / G), j % G);
      const double ej = c.atol + c.rtol * fabs(yj);
      const double r = fmax(srur * fabs(yj), r0 / ej);
      double yp[R], ft[R], col[R];
      if (c.order == 1) {
#pragma unroll
        for (int q = 0; q < R; ++q) yp[q] = (RW::valid(ln, q) && RW::row(ln, q) == j) ? yj + r : y[q];
        Base::template dydt<G, R>(c, t, pr, yp, ft);
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] = (ft[q] - f0[q]) / r;
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] = 0.0;
#pragma unroll 1
        for (int k = 0; k < c.order; ++k) {
          double xk, wk;
          fd_stencil(c.order, k, xk, wk);
#pragma unroll
          for (int q = 0; q < R; ++q) yp[q] = (RW::valid(ln, q) && RW::row(ln, q) == j) ? yj + xk * r : y[q];
          Base::template dydt<G, R>(c, t, pr, yp, ft);
#pragma unroll
          for (int q = 0; q < R; ++q) col[q] += wk * ft[q];
        }
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] /= r;
      }
      put(j, col);
    }
  }

  // Jacobian parked in the group's LDS (rows or columns, as the base mechanism parks it)
  template <int G, int R>
  __device__ __forceinline__ static void jacob(Ctx& c, double t, double pr, const double (&y)[R]) {
    using RW = Rows<N, G, R>;
    const int ln = Grp<G>::lane();
    columns<G, R>(c, t, pr, y, [&](int j, const double (&col)[R]) {
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (RW::valid(ln, q)) c.jac[jidx<Base>(RW::row(ln, q), j)] = col[q];
    });
    group_lds_sync();
  }

  // Jacobian in registers (J[q][j] = d f_row / d y_j)
  template <int G, int R>
  __device__ __forceinline__ static void jacob(Ctx& c, double t, double pr, const double (&y)[R], double (&J)[R][N]) {
    columns<G, R>(c, t, pr, y, [&](int j, const double (&col)[R]) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
#pragma unroll
        for (int k = 0; k < N; ++k)
          if (k == j) J[q][k] = col[q];
      }
    });
  }
};

}  // namespace acc
