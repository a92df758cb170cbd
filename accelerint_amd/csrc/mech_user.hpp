// A user mechanism compiled into the integrator: adapts pyJac-style device
// callbacks (dydt / eval_jacob over one condition's arrays, the contract of
// include/accelerint_mechanism.h, after examples/van_der_pol/dydt.cuh:26-28
// and jacob.cuh:23-24) to the lane-group layout.
//
// The user's sources arrive as one include list (ACCELERINT_USER_SOURCES, a
// file written by the build) and are compiled into this translation unit.
// Lane groups by size: up to 4 states one condition per lane (its arrays in
// registers), up to 16 a 16-lane group, up to 64 a wavefront.  In a group the
// callbacks are serial code for one condition: the group's lanes put their
// rows of y into the group's LDS slice, lane 0 runs the callback there, and
// each lane reads back its rows of dy; the Jacobian stays column-major in the
// group's LDS (jac[i + j N]), where the integrator reads it.
#pragma once

#include "accelerint_mechanism.h"
#include "mechanism.h"

#include ACCELERINT_USER_SOURCES

#include "radau_core.hpp"

#ifndef NSP
#error "mechanism.h must define NSP, the system size"
#endif

namespace acc {

constexpr int kUserN = NSP;
static_assert(kUserN >= 1 && kUserN <= 64, "user mechanisms of 1 to 64 states are supported");
#ifdef ACCELERINT_NO_ANALYTIC_JACOBIAN
constexpr bool kUserHasJacobian = false;
#else
constexpr bool kUserHasJacobian = true;
#endif
constexpr int kUserG = kUserN <= 4 ? 1 : (kUserN <= 16 ? 16 : 64);
constexpr int kUserR = kUserG == 1 ? kUserN : 1;
constexpr int kUserBlock = kUserG == 64 ? 256 : (kUserG == 16 ? 128 : 256);

struct MechUser {
  static constexpr int N = kUserN;
  static constexpr bool kJacInLds = kUserG > 1;
  static constexpr bool kJacColMajor = true;
  struct Params {};
  // per group: y, dy, the parameter and the Jacobian (N x N)
  __host__ __device__ static size_t group_doubles() { return kJacInLds ? (size_t)2 * N + 2 + (size_t)N * N : 0; }
  static size_t lds_bytes(const Params&, int groups) {
    return (size_t)groups * group_doubles() * sizeof(double);
  }
  __device__ __forceinline__ static void block_init(const Params&, double*) {}

  struct Ctx {
    double* yb = nullptr;
    double* dyb = nullptr;
    double* var = nullptr;
    double* jac = nullptr;
    __device__ Ctx(const Params& p, int g, double* lds) : Ctx(p, lds, lds + (size_t)g * group_doubles()) {}
    __device__ Ctx(const Params&, const double*, double* group) {
      if constexpr (kJacInLds) {
        yb = group;
        dyb = yb + N;
        var = dyb + N;
        jac = var + 2;
      }
    }
  };

  // Rows of y into the group's LDS slice, then lane 0 runs `call` there.
  template <int G, int R, class Call>
  __device__ __forceinline__ static void on_lane0(Ctx& c, double pr, const double (&y)[R], Call&& call) {
    const int ln = Grp<G>::lane();
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (ln + G * q < N) c.yb[ln + G * q] = y[q];
    if (ln == 0) c.var[0] = pr;
    group_lds_sync();
    if (ln == 0) {
      const mechanism_memory m{c.yb, c.dyb, c.var, c.jac};
      call(m);
    }
    group_lds_sync();
  }

  template <int G, int R>
  __device__ __forceinline__ static void dydt(Ctx& c, double t, double pr, const double (&y)[R], double (&f)[R]) {
    if constexpr (G == 1) {
      double yy[N], dd[N];
#pragma unroll
      for (int i = 0; i < N; ++i) yy[i] = y[i];
      const mechanism_memory m{yy, dd, &pr, nullptr};
      ::dydt(t, pr, yy, dd, &m);
#pragma unroll
      for (int i = 0; i < N; ++i) f[i] = dd[i];
    } else {
      on_lane0<G, R>(c, pr, y, [&](const mechanism_memory& m) { ::dydt(t, pr, c.yb, c.dyb, &m); });
      const int ln = Grp<G>::lane();
#pragma unroll
      for (int q = 0; q < R; ++q) f[q] = (ln + G * q < N) ? c.dyb[ln + G * q] : 0.0;
      group_lds_sync();  // every lane has read dy before the next call writes it
    }
  }

  // Jacobian into the group's LDS, column-major (kJacInLds).
  template <int G, int R>
  __device__ __forceinline__ static void jacob(Ctx& c, double t, double pr, const double (&y)[R]) {
    if constexpr (kUserHasJacobian) {
      on_lane0<G, R>(c, pr, y, [&](const mechanism_memory& m) { ::eval_jacob(t, pr, c.yb, c.jac, &m); });
    }
  }

  // Jacobian in registers (one condition per lane): J[q][j] = d f_q / d y_j.
  template <int G, int R>
  __device__ __forceinline__ static void jacob(Ctx&, double t, double pr, const double (&y)[R], double (&J)[R][N]) {
    if constexpr (kUserHasJacobian && G == 1) {
      double yy[N], jj[N * N];
#pragma unroll
      for (int i = 0; i < N; ++i) yy[i] = y[i];
      const mechanism_memory m{yy, nullptr, &pr, jj};
      ::eval_jacob(t, pr, yy, jj, &m);
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int j = 0; j < N; ++j) J[q][j] = jj[q + j * N];
    }
  }
};

}  // namespace acc
