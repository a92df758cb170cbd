// Batched Radau IIA (order 5) for gfx950: one condition per lane group.
//
// Layout: a condition is integrated by a group of G lanes inside one
// wavefront (G divides 64).  Lane l of the group owns rows r = l + G*q,
// q < R, of every row-indexed quantity: the state y, the stage vectors, and
// full rows of the Jacobian and of the two iteration matrices.  Matrix rows
// live in VGPRs with compile-time column indices, so the dense LU and the
// triangular solves are straight-line FMA code; the only cross-lane traffic is
// the pivot search (group argmax), the pivot-row broadcast and the scalar
// reductions of the error norms.  Every scalar of the step-size controller is
// group-uniform, so each group runs its own control flow.
//
// The algorithm follows the reference's CPU integrator radau2a/radau2a.c
// (integrate :520-736) step for step; the LU follows LAPACK dgetf2/zgetf2
// semantics (partial pivoting, first maximum, |Re|+|Im| for complex), done with
// implicit row interchanges: rows never move between lanes, each row records
// the LAPACK position it would occupy so ties break exactly as LAPACK would.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mlp.hpp"

namespace acc {

// ---- control constants: radau2a.c:37-66 ------------------------------------
constexpr int kMaxNoSteps = 200000;
constexpr int kNewtonMaxit = 8;
constexpr double kRoundoff = 2.220446049250313080847e-16;  // DBL_EPSILON
constexpr double kFacMin = 0.2;
constexpr double kFacMax = 8.0;
constexpr double kFacSafe = 0.9;
constexpr double kFacRej = 0.1;
constexpr double kThetaMin = 0.001;
constexpr double kNewtonTol = 0.03;
constexpr double kQmin = 1.0;
constexpr double kQmax = 1.2;
constexpr int kMaxConsecutiveErrs = 5;
constexpr double kDblMin = 2.2250738585072014e-308;
// Mixed precision with the workspace LU (more than 64 states) only, no
// counterpart in the reference: an FP32-factor run that needs more than this
// many steps for one global step gives up with the max-steps code, which
// hands the condition to the FP64 pass.  A 112-state condition whose FP32
// Newton iteration converges only at tiny H would otherwise crawl towards
// kMaxNoSteps (minutes per condition); at up to 64 states steps are cheap
// and long conditions are legitimate, so the reference's limit applies.
constexpr int kMixedMaxSteps = 10000;

// ---- Radau IIA(5) tableau, as published by Hairer & Wanner (RADAU5) --------
// Same digits as radau2a.c:101-231; every value is re-derived from closed
// forms by the test suite.
constexpr double rkA00 = 1.968154772236604258683861429918299e-1;
constexpr double rkA01 = -6.55354258501983881085227825696087e-2;
constexpr double rkA02 = 2.377097434822015242040823210718965e-2;
constexpr double rkA10 = 3.944243147390872769974116714584975e-1;
constexpr double rkA11 = 2.920734116652284630205027458970589e-1;
constexpr double rkA12 = -4.154875212599793019818600988496743e-2;
constexpr double rkA20 = 3.764030627004672750500754423692808e-1;
constexpr double rkA21 = 5.124858261884216138388134465196080e-1;
constexpr double rkA22 = 1.111111111111111111111111111111111e-1;
constexpr double rkC0 = 1.550510257216821901802715925294109e-1;
constexpr double rkC1 = 6.449489742783178098197284074705891e-1;
constexpr double rkC2 = 1.0;
constexpr double rkE0 = 0.05;
constexpr double rkE1 = -10.04880939982741556246032950764708 * 0.05;
constexpr double rkE2 = 1.382142733160748895793662840980412 * 0.05;
constexpr double rkE3 = -0.3333333333333333333333333333333333 * 0.05;
constexpr double rkGamma = 3.637834252744495732208418513577775;
constexpr double rkAlpha = 2.681082873627752133895790743211112;
constexpr double rkBeta = 3.050430199247410569426377624787569;
constexpr double rkT00 = 9.443876248897524148749007950641664e-2;
constexpr double rkT01 = -1.412552950209542084279903838077973e-1;
constexpr double rkT02 = -3.00291941051474244918611170890539e-2;
constexpr double rkT10 = 2.502131229653333113765090675125018e-1;
constexpr double rkT11 = 2.041293522937999319959908102983381e-1;
constexpr double rkT12 = 3.829421127572619377954382335998733e-1;
constexpr double rkT20 = 1.0;
constexpr double rkT21 = 1.0;
constexpr double rkT22 = 0.0;
constexpr double rkTiAi00 = 1.520148562492775501049204957366528e+1;
constexpr double rkTiAi01 = 1.192055789400527921212348994770778;
constexpr double rkTiAi02 = 1.903956760517560343018332287285119;
constexpr double rkTiAi10 = -9.669512977505946748632625374449567;
constexpr double rkTiAi11 = -8.724028436822336183071773193986487;
constexpr double rkTiAi12 = 3.096043239482439656981667712714881;
constexpr double rkTiAi20 = -1.409513259499574544876303981551774e+1;
constexpr double rkTiAi21 = 5.895975725255405108079130152868952;
constexpr double rkTiAi22 = -1.441236197545344702389881889085515e-1;
constexpr double rkELO = 4.0;


// Return codes: radau2a/radau2a_props.h:30-39.
enum : int {
  EC_success = 0,
  EC_consecutive_steps = 1,
  EC_max_steps_exceeded = 2,
  EC_h_plus_t_equals_h = 3,
  EC_newton_max_iterations_exceeded = 4,
};

// Per-condition event counters (algorithmic-work accounting); the order
// matches the oracle's.
enum : int {
  CNT_STEP = 0, CNT_ACCEPT, CNT_REJECT, CNT_NEWTON_FAIL, CNT_LU, CNT_LU_FAIL,
  CNT_NEWTON, CNT_F, CNT_JAC, CNT_ES, NCNT
};

struct SolverParams {
  double atol;
  double rtol;
  int const_time_step;
  MlpView mlp;    // learned Newton start of each global step's first step (on = 0: zero start)
  StartLog log;   // training-sample log (cap = 0: off)
  // per-group global workspace of the large systems (memory-resident factors,
  // parked Jacobian): group g of the grid at ws + g * ws_bytes, for at most
  // ws_groups groups (0: none)
  char* ws = nullptr;
  size_t ws_bytes = 0;
  int ws_groups = 0;
};

// ---- lane-group primitives ---------------------------------------------------
template <int G>
struct Grp {
  static_assert(G >= 1 && G <= 64 && (G & (G - 1)) == 0, "group width must be a power of two");
  __device__ __forceinline__ static int lane() { return (int)(__lane_id() & (G - 1)); }

  __device__ __forceinline__ static double bcast(double v, int src) {
    if constexpr (G == 1) {
      return v;
    } else if constexpr (G == 64) {
      // src is wave-uniform: read it through SGPRs.
      int s = __builtin_amdgcn_readfirstlane(src);
      int lo = __builtin_amdgcn_readlane(__double2loint(v), s);
      int hi = __builtin_amdgcn_readlane(__double2hiint(v), s);
      return __hiloint2double(hi, lo);
    } else {
      return __shfl(v, src, G);
    }
  }
  __device__ __forceinline__ static float bcast(float v, int src) {
    if constexpr (G == 1) {
      return v;
    } else if constexpr (G == 64) {
      int s = __builtin_amdgcn_readfirstlane(src);
      return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), s));
    } else {
      return __shfl(v, src, G);
    }
  }
  __device__ __forceinline__ static int bcast_i(int v, int src) {
    if constexpr (G == 1) {
      return v;
    } else if constexpr (G == 64) {
      int s = __builtin_amdgcn_readfirstlane(src);
      return __builtin_amdgcn_readlane(v, s);
    } else {
      return __shfl(v, src, G);
    }
  }
  // per-lane source (ds_bpermute)
  __device__ __forceinline__ static double gather(double v, int src) {
    if constexpr (G == 1) {
      return v;
    } else {
      return __shfl(v, src, G);
    }
  }
  __device__ __forceinline__ static double xor_(double v, int m) { return __shfl_xor(v, m, G); }
  __device__ __forceinline__ static float xor_(float v, int m) { return __shfl_xor(v, m, G); }
  __device__ __forceinline__ static int xor_i(int v, int m) { return __shfl_xor(v, m, G); }

  // Butterfly all-reduce: partners add the same two operands, so every lane
  // of the group ends with a bit-identical result.
  __device__ __forceinline__ static double sum(double v);
  // two sums side by side: the same operations as two calls of sum, their
  // dependent chains overlapped
  __device__ __forceinline__ static void sum2(double& a, double& b);
  __device__ __forceinline__ static void sum3(double& a, double& b, double& c);
};

// Row ownership helpers.
template <int N, int G, int R>
struct Rows {
  static_assert(G * R >= N, "group too small for system size");
  __device__ __forceinline__ static int row(int ln, int q) { return ln + G * q; }
  __device__ __forceinline__ static bool valid(int ln, int q) { return ln + G * q < N; }
};

// Where a mechanism parks its Jacobian in LDS: rows (jac[r*N + j], the
// built-in networks) or columns (jac[r + j*N], the reference's column-major
// callback layout, which user mechanisms write directly).
template <class M, class = void>
struct JacColMajor : std::false_type {};
template <class M>
struct JacColMajor<M, std::void_t<decltype(M::kJacColMajor)>> : std::integral_constant<bool, M::kJacColMajor> {};
// Leading dimension of a column-major parked Jacobian (default N).
template <class M, class = void>
struct JacLd : std::integral_constant<int, M::N> {};
template <class M>
struct JacLd<M, std::void_t<decltype(M::kJacLd)>> : std::integral_constant<int, M::kJacLd> {};
// Mechanisms whose jacob takes a third template argument, the batch width of
// its accumulation, with preferred widths for FP32 and FP64 factor kernels.
template <class M, class = void>
struct JacBatched : std::false_type {};
template <class M>
struct JacBatched<M, std::void_t<decltype(M::kJacBatchFP32)>> : std::true_type {};
template <class Mech>
__device__ __forceinline__ constexpr int jidx(int r, int j) {
  return JacColMajor<Mech>::value ? r + j * JacLd<Mech>::value : r * Mech::N + j;
}

// Select x[q] for a runtime q without dynamic register indexing.
template <int R, class T>
__device__ __forceinline__ T sel(const T (&x)[R], int q) {
  T v = x[0];
#pragma unroll
  for (int i = 1; i < R; ++i) v = (q == i) ? x[i] : v;
  return v;
}

// Packed pivot-row table: entry k = row that was the pivot at elimination step k.
template <int N>
struct Perm {
  uint32_t w[(N + 3) / 4];
  __device__ __forceinline__ void set(int k, int row) {
    const int s = 8 * (k & 3);
    w[k >> 2] = (w[k >> 2] & ~(0xffu << s)) | ((uint32_t)row << s);
  }
  __device__ __forceinline__ int get(int k) const { return (int)((w[k >> 2] >> (8 * (k & 3))) & 0xffu); }
};

// Smallest normal number of the matrix scalar type (LAPACK's sfmin test).
template <class T>
__device__ __forceinline__ constexpr T min_normal() {
  if constexpr (std::is_same<T, float>::value) return 1.17549435082228750797e-38f;
  else return kDblMin;
}

// Reciprocal of the pivot: IEEE division in FP64 (bit-compatible with the
// oracle's LAPACK semantics); in FP32 (mixed precision, no bit parity) the
// hardware reciprocal refined by one Newton step, within 1 ulp.
template <class T>
__device__ __forceinline__ T recip(T x) {
  if constexpr (std::is_same<T, float>::value) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
  } else {
    return 1.0 / x;
  }
}

// Smith's complex reciprocal 1/(c + i d).
template <class T>
__device__ __forceinline__ void crecip(T c, T d, T& re, T& im) {
  if constexpr (std::is_same<T, float>::value) {
    // FP32 factors: the same formula with refined hardware reciprocals
    const bool cd = fabsf(c) >= fabsf(d);
    const float a = cd ? c : d, b = cd ? d : c;
    const float r = b * recip(a), den = a + b * r, iden = recip(den);
    re = cd ? iden : r * iden;
    im = cd ? -r * iden : -iden;
  } else {
    // selected operands, not branches: in lane groups narrower than a wavefront
    // both sides would run, and the two quotients overlap
    const bool cd = fabs(c) >= fabs(d);
    const T a = cd ? c : d, b = cd ? d : c;
    const T r = b / a, den = a + b * r;
    const T iden = T(1) / den, rden = r / den;
    re = cd ? iden : rden;
    im = cd ? -rden : -iden;
  }
}

// DPP lane exchanges inside a 16-lane row: quad_perm [1,0,3,2] (xor 1),
// quad_perm [2,3,0,1] (xor 2), row_half_mirror (i <-> 7 - i in each 8) and
// row_mirror (i <-> 15 - i).  Applied in that order, a commutative pairwise
// combine leaves every lane of the row with the combination of all 16.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_t(float v) {
  return __int_as_float(dpp_i<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_t(double v) {
  return __hiloint2double(dpp_i<CTRL>(__double2hiint(v)), dpp_i<CTRL>(__double2loint(v)));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
// (value, key) order of the pivot search: larger value, then smaller key.
// Cross-row exchanges of a 64-lane wave on the VALU (gfx950
// v_permlane16_swap / v_permlane32_swap).  Called with a == b == v:
// swap_row_pairs leaves a = v of rows (0, 0, 2, 2) and b = v of rows
// (1, 1, 3, 3) in rows 0..3; swap_halves leaves a = v of lanes 0-31 and
// b = v of lanes 32-63 in both halves.
__device__ __forceinline__ void swap_row_pairs(int& a, int& b) {
  const auto r = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
  a = (int)r[0];
  b = (int)r[1];
}
__device__ __forceinline__ void swap_halves(int& a, int& b) {
  const auto r = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
  a = (int)r[0];
  b = (int)r[1];
}
__device__ __forceinline__ void swap_row_pairs(float& a, float& b) {
  int x = __float_as_int(a), y = __float_as_int(b);
  swap_row_pairs(x, y);
  a = __int_as_float(x);
  b = __int_as_float(y);
}
__device__ __forceinline__ void swap_halves(float& a, float& b) {
  int x = __float_as_int(a), y = __float_as_int(b);
  swap_halves(x, y);
  a = __int_as_float(x);
  b = __int_as_float(y);
}
__device__ __forceinline__ void swap_row_pairs(double& a, double& b) {
  int al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
  swap_row_pairs(al, bl);
  swap_row_pairs(ah, bh);
  a = __hiloint2double(ah, al);
  b = __hiloint2double(bh, bl);
}
__device__ __forceinline__ void swap_halves(double& a, double& b) {
  int al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
  swap_halves(al, bl);
  swap_halves(ah, bh);
  a = __hiloint2double(ah, al);
  b = __hiloint2double(bh, bl);
}

// Bitwise, not short-circuit, so the exchange stays branch-free.
template <class T>
__device__ __forceinline__ void argmax_merge(T& bv, int& bkey, T ov, int ok) {
  const bool better = (ov > bv) | ((ov == bv) & (ok < bkey));
  bv = better ? ov : bv;
  bkey = better ? ok : bkey;
}

// Argmax over the group of (value, key) with key = (LAPACK position << 8) | row;
// larger value wins, equal values go to the smaller position (first maximum).
// The order is total on non-NaN values, so every pairing network returns the
// same winner: 16- and 64-lane groups use DPP within rows, other widths an
// xor butterfly.
template <int G, class T>
__device__ __forceinline__ void group_argmax(T& bv, int& bkey) {
  if constexpr (G == 16) {
    argmax_merge(bv, bkey, dpp_t<kDppXor1>(bv), dpp_i<kDppXor1>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppXor2>(bv), dpp_i<kDppXor2>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppHalfMirror>(bv), dpp_i<kDppHalfMirror>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppMirror>(bv), dpp_i<kDppMirror>(bkey));
  } else if constexpr (G == 64) {
    // DPP within each 16-lane row, then the row winners joined by the VALU
    // lane swaps (row pairs 0|1 and 2|3, then halves), which replace two
    // ds_bpermute round trips per exchange.  Every lane merges (lower, upper)
    // in that order, so all 64 lanes end with the same winner.  (Two other
    // ways to join the rows picked wrong pivots on gfx950 and are not used:
    // merging the four row winners after reading them into scalar registers,
    // and DPP row_bcast:15 / row_bcast:31 with row masks.)
    argmax_merge(bv, bkey, dpp_t<kDppXor1>(bv), dpp_i<kDppXor1>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppXor2>(bv), dpp_i<kDppXor2>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppHalfMirror>(bv), dpp_i<kDppHalfMirror>(bkey));
    argmax_merge(bv, bkey, dpp_t<kDppMirror>(bv), dpp_i<kDppMirror>(bkey));
    {
      T lo = bv, hi = bv;
      int klo = bkey, khi = bkey;
      swap_row_pairs(lo, hi);
      swap_row_pairs(klo, khi);
      bv = lo;
      bkey = klo;
      argmax_merge(bv, bkey, hi, khi);
    }
    {
      T lo = bv, hi = bv;
      int klo = bkey, khi = bkey;
      swap_halves(lo, hi);
      swap_halves(klo, khi);
      bv = lo;
      bkey = klo;
      argmax_merge(bv, bkey, hi, khi);
    }
  } else {
#pragma unroll
    for (int m = 1; m < G; m <<= 1) argmax_merge(bv, bkey, Grp<G>::xor_(bv, m), Grp<G>::xor_i(bkey, m));
  }
}


// Pivot search of the register LU at G = 64, one row per lane (wave_pivot2, row = lane):
// the first maximum of the magnitudes v over the active lanes in LAPACK's row
// order (pos), as a wave-uniform lane, or -1 if no active lane holds a
// comparable value (every candidate NaN).  The magnitudes are compared as
// integers (non-negative floats order as their bits); only the leading 32 bits
// go through the lane exchanges, one v_max_u32 per exchange, and the lanes that
// attain the maximum come out of one compare as a scalar mask.  Lanes that agree
// in those bits, which is rare, are compared one by one in full.  Against an
// exchange of (value, key) pairs joined through scalar mask logic this is ~20
// instead of 84 instructions per FP64 search.
__device__ __forceinline__ unsigned mag_hi(float v) { return __float_as_uint(v); }
__device__ __forceinline__ unsigned mag_hi(double v) { return (unsigned)__double2hiint(v); }
__device__ __forceinline__ unsigned max_u(unsigned a, unsigned b) { return a > b ? a : b; }
template <int CTRL>
__device__ __forceinline__ unsigned dpp_max_u(unsigned v) {
  return max_u(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false));
}
// The lane among cand, the lanes whose keys equal the maximum m: decided by the
// full magnitudes, then by the row order.
template <class T>
__device__ __forceinline__ int wave_pivot_tie(T v, int pos, unsigned m, unsigned long long cand) {
  if (m == 0) return -1;
  int lane = -1;
  T bv = T(0);
  int best = 0;
  while (cand) {
    const int l = (int)__builtin_ctzll(cand);
    cand &= cand - 1;
    const T w = Grp<64>::bcast(v, l);
    const int q = __builtin_amdgcn_readlane(pos, l);
    if (lane < 0 || w > bv || (w == bv && q < best)) {
      bv = w;
      best = q;
      lane = l;
    }
  }
  return __builtin_amdgcn_readfirstlane(lane);
}
// Two searches side by side: each is one chain of dependent lane exchanges.
template <class T>
__device__ __forceinline__ void wave_pivot2(T v, int pos, bool act, T v2, int pos2, bool act2, int& lane, int& lane2) {
  const unsigned key = act && v == v ? mag_hi(v) + 1u : 0u;  // 0: no candidate
  const unsigned key2 = act2 && v2 == v2 ? mag_hi(v2) + 1u : 0u;
  unsigned m = dpp_max_u<kDppXor1>(key), m2 = dpp_max_u<kDppXor1>(key2);
  m = dpp_max_u<kDppXor2>(m), m2 = dpp_max_u<kDppXor2>(m2);
  m = dpp_max_u<kDppHalfMirror>(m), m2 = dpp_max_u<kDppHalfMirror>(m2);
  m = dpp_max_u<kDppMirror>(m), m2 = dpp_max_u<kDppMirror>(m2);
  int x = (int)m, y = (int)m, x2 = (int)m2, y2 = (int)m2;
  swap_row_pairs(x, y);
  swap_row_pairs(x2, y2);
  x = y = (int)max_u((unsigned)x, (unsigned)y);
  x2 = y2 = (int)max_u((unsigned)x2, (unsigned)y2);
  swap_halves(x, y);
  swap_halves(x2, y2);
  m = (unsigned)__builtin_amdgcn_readfirstlane((int)max_u((unsigned)x, (unsigned)y));
  m2 = (unsigned)__builtin_amdgcn_readfirstlane((int)max_u((unsigned)x2, (unsigned)y2));
  const unsigned long long cand = __builtin_amdgcn_ballot_w64(key == m);
  const unsigned long long cand2 = __builtin_amdgcn_ballot_w64(key2 == m2);
  lane = (int)__builtin_ctzll(cand);  // (the lane that holds the maximum: never empty)
  lane2 = (int)__builtin_ctzll(cand2);
  const unsigned long long tie = cand & (cand - 1), tie2 = cand2 & (cand2 - 1);
  if (__builtin_expect((tie | tie2) != 0, 0)) {
    if (tie) lane = wave_pivot_tie(v, pos, m, cand);
    if (tie2) lane2 = wave_pivot_tie(v2, pos2, m2, cand2);
  }
}

// Tests of a wave-uniform pivot on its bits, in scalar registers.
__device__ __forceinline__ bool is_zero(float v) { return (__float_as_uint(v) & 0x7fffffffu) == 0; }
__device__ __forceinline__ bool is_zero(double v) {
  return (((unsigned)__double2hiint(v) & 0x7fffffffu) | (unsigned)__double2loint(v)) == 0;
}
__device__ __forceinline__ bool is_subnormal_or_zero(double v) {
  return ((unsigned)__double2hiint(v) & 0x7fffffffu) < 0x00100000u;
}

// Keeps a value where it is computed: the compiler neither moves its
// computation past this point nor recomputes or specializes it later (v: a
// vector register, s: a scalar one, for wave-uniform values).
template <class T>
__device__ __forceinline__ void pin(T& v) {
  __asm__ volatile("" : "+v"(v));
}
template <class T>
__device__ __forceinline__ void pin_s(T& v) {
  v = (T)__builtin_amdgcn_readfirstlane((int)v);
  __asm__ volatile("" : "+s"(v));
}
// Columns whose pivot-row entries are in scalar registers at once (the
// updates of one chunk are pinned before the next one's): more of them at once
// overflow the 102 scalar registers, and every spilled broadcast costs two
// lane moves.
constexpr int kBcastChunk = 8;

// Group all-reduce of a sum.  16- and 64-lane groups: DPP pairs within rows
// (each pair adds the same two operands, so the lanes of a row agree bit for
// bit), then for 64 the four row sums in a fixed order from SGPRs; other
// widths: xor butterfly.
template <int G>
__device__ __forceinline__ double Grp<G>::sum(double v) {
  if constexpr (G == 16 || G == 64) {
    v += dpp_t<kDppXor1>(v);
    v += dpp_t<kDppXor2>(v);
    v += dpp_t<kDppHalfMirror>(v);
    v += dpp_t<kDppMirror>(v);
    if constexpr (G == 64) v = (bcast(v, 0) + bcast(v, 16)) + (bcast(v, 32) + bcast(v, 48));
  } else {
#pragma unroll
    for (int m = 1; m < G; m <<= 1) v += xor_(v, m);
  }
  return v;
}

template <int G>
__device__ __forceinline__ void Grp<G>::sum2(double& a, double& b) {
  if constexpr (G == 16 || G == 64) {
    double x = dpp_t<kDppXor1>(a), z = dpp_t<kDppXor1>(b);
    a += x;
    b += z;
    x = dpp_t<kDppXor2>(a), z = dpp_t<kDppXor2>(b);
    a += x;
    b += z;
    x = dpp_t<kDppHalfMirror>(a), z = dpp_t<kDppHalfMirror>(b);
    a += x;
    b += z;
    x = dpp_t<kDppMirror>(a), z = dpp_t<kDppMirror>(b);
    a += x;
    b += z;
    if constexpr (G == 64) {
      a = (bcast(a, 0) + bcast(a, 16)) + (bcast(a, 32) + bcast(a, 48));
      b = (bcast(b, 0) + bcast(b, 16)) + (bcast(b, 32) + bcast(b, 48));
    }
  } else {
    a = sum(a);
    b = sum(b);
  }
}

template <int G>
__device__ __forceinline__ void Grp<G>::sum3(double& a, double& b, double& c) {
  if constexpr (G == 16 || G == 64) {
    double x = dpp_t<kDppXor1>(a), z = dpp_t<kDppXor1>(b), w = dpp_t<kDppXor1>(c);
    a += x;
    b += z;
    c += w;
    x = dpp_t<kDppXor2>(a), z = dpp_t<kDppXor2>(b), w = dpp_t<kDppXor2>(c);
    a += x;
    b += z;
    c += w;
    x = dpp_t<kDppHalfMirror>(a), z = dpp_t<kDppHalfMirror>(b), w = dpp_t<kDppHalfMirror>(c);
    a += x;
    b += z;
    c += w;
    x = dpp_t<kDppMirror>(a), z = dpp_t<kDppMirror>(b), w = dpp_t<kDppMirror>(c);
    a += x;
    b += z;
    c += w;
    if constexpr (G == 64) {
      a = (bcast(a, 0) + bcast(a, 16)) + (bcast(a, 32) + bcast(a, 48));
      b = (bcast(b, 0) + bcast(b, 16)) + (bcast(b, 32) + bcast(b, 48));
      c = (bcast(c, 0) + bcast(c, 16)) + (bcast(c, 32) + bcast(c, 48));
    }
  } else {
    a = sum(a);
    b = sum(b);
    c = sum(c);
  }
}

// ---- real LU (dgetf2 semantics, implicit interchanges) ---------------------
// On exit a[q][*] holds row r's L multipliers (columns < pos[q]) and U entries
// (columns >= pos[q]); pos[q] is the elimination step at which row r was the
// pivot; perm.get(k) is the pivot row of step k; rd[q] = 1 / U(r, pos[q]).
// info = first step (1-based) with an exactly zero pivot, 0 otherwise.
//
// Rows that do not take part in step k (the pivot row, rows already
// eliminated, padding rows) get a zero multiplier, so the update is
// branch-free and each pivot-row entry is broadcast just before the column
// update that consumes it.
template <int N, int G, int R, class T>
__device__ __forceinline__ void lu_init(int (&pos)[R], T (&rd)[R], int& info) {
  const int ln = Grp<G>::lane();
#pragma unroll
  for (int q = 0; q < R; ++q) {
    pos[q] = Rows<N, G, R>::valid(ln, q) ? Rows<N, G, R>::row(ln, q) : -1;
    rd[q] = T(0);
  }
  info = 0;
}

// Elimination step k of the real and the complex LU together, a wavefront per
// pair of matrices and a row of each per lane (k a compile-time constant after
// unrolling): for each matrix the operations of lu_real_step and lu_cplx_step
// below in the same order.  Bound by the issue of a lane move per broadcast
// pivot-row word and the step's chain search -> reciprocal -> multiplier; the
// two chains are independent and are issued side by side.  What a step leaves
// behind (multipliers, reciprocals, positions, pivot rows, updated columns) is
// pinned to the step, column after column: left alone, the compiler delayed the
// selects and updates of each step past the next one's branches, which kept up
// to 54 broadcasts alive in scalar registers (spilled by two lane moves each)
// and gave every step scratch slots.  Order 54, cycles for the pair of
// factorizations with one wavefront per SIMD, one matrix after the other ->
// together: FP64 181600 -> 178700, FP32 119100 -> 107700; 65536 conditions of
// one global step with FP32 factors 155.6 -> 149.1 ms, 32768 in FP64
// 103.0 -> 102.6 ms.  (In FP64 the schedule is cut around the updates: without
// the cuts 176100 cycles, but the longer live ranges cost the kernel that holds
// all three networks 1%.  Filling each chain's waits with the other matrix's
// column updates was slower, 117000 cycles in FP32: a broadcast used at once
// waits longer than the chain does.)
template <int N, class T>
__device__ __forceinline__ void wave_lu_step(const int k, T (&a)[N], int& pos, Perm<N>& perm, T& rd, int& info,
                                             T (&ar)[N], T (&ai)[N], int& pos2, Perm<N>& perm2, T& rdr, T& rdi,
                                             int& info2) {
  const int ln = Grp<64>::lane();
  int win, win2;
  wave_pivot2(fabs(a[k]), pos, pos >= k, fabs(ar[k]) + fabs(ai[k]), pos2, pos2 >= k, win, win2);
  const int plane = win & 63, plane2 = win2 & 63;
  const int prow = win >= 0 ? win : 0xff, prow2 = win2 >= 0 ? win2 : 0xff;
  const int pp = __builtin_amdgcn_readlane(pos, plane), pp2 = __builtin_amdgcn_readlane(pos2, plane2);
  const T piv = Grp<64>::bcast(a[k], plane);
  const T pr_ = Grp<64>::bcast(ar[k], plane2);
  const T pi_ = Grp<64>::bcast(ai[k], plane2);
  const T rp = recip(piv);
  T rr, ri;
  crecip(pr_, pi_, rr, ri);
  const int ppos = win >= 0 ? pp : 0x7fffff, ppos2 = win2 >= 0 ? pp2 : 0x7fffff;
  perm.set(k, prow);
  perm2.set(k, prow2);
  const bool nz = !is_zero(piv), nz2 = !(is_zero(pr_) && is_zero(pi_));
  info = !nz && info == 0 ? k + 1 : info;
  info2 = !nz2 && info2 == 0 ? k + 1 : info2;
  const bool is_piv = ln == prow, is_piv2 = ln == prow2;
  pos = is_piv ? k : (pos == k ? ppos : pos);  // LAPACK swaps rows k and ppos
  pos2 = is_piv2 ? k : (pos2 == k ? ppos2 : pos2);
  T lq = a[k] * rp;
  // LAPACK divides instead of scaling by the reciprocal when |pivot| < sfmin
  // (FP64 path only; the FP32 factors need no such care)
  if constexpr (std::is_same<T, double>::value)
    if (__builtin_expect(is_subnormal_or_zero(piv), 0)) lq = a[k] / piv;
  rd = is_piv ? (nz ? rp : T(0)) : rd;
  rdr = is_piv2 ? (nz2 ? rr : T(0)) : rdr;
  rdi = is_piv2 ? (nz2 ? ri : T(0)) : rdi;
  const bool act = nz && pos > k, act2 = nz2 && pos2 > k;
  a[k] = act ? lq : a[k];
  T l = act ? -lq : T(-0.0);
  const T xr = ar[k], xi = ai[k];
  const T vr = xr * rr - xi * ri;
  const T vi = xr * ri + xi * rr;
  ar[k] = act2 ? vr : xr;
  ai[k] = act2 ? vi : xi;
  T lr = act2 ? vr : T(0), li = act2 ? vi : T(0);
  pin_s(perm.w[k >> 2]);
  pin_s(perm2.w[k >> 2]);
  pin(info);
  pin(info2);
  pin(pos);
  pin(pos2);
  pin(rd);
  pin(rdr);
  pin(rdi);
  pin(a[k]);
  pin(l);
  pin(ar[k]);
  pin(ai[k]);
  pin(lr);
  pin(li);
  if constexpr (std::is_same<T, double>::value) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j0 = k + 1; j0 < N; j0 += kBcastChunk) {
    T u[kBcastChunk];
#pragma unroll
    for (int j = j0; j < j0 + kBcastChunk; ++j)
      if (j < N) u[j - j0] = Grp<64>::bcast(a[j], plane);
#pragma unroll
    for (int j = j0; j < j0 + kBcastChunk; ++j)
      if (j < N) {
        a[j] = fma(l, u[j - j0], a[j]);
        pin(a[j]);
      }
  }
#pragma unroll
  for (int j0 = k + 1; j0 < N; j0 += kBcastChunk) {
    T ur[kBcastChunk], ui[kBcastChunk];
#pragma unroll
    for (int j = j0; j < j0 + kBcastChunk; ++j)
      if (j < N) {
        ur[j - j0] = Grp<64>::bcast(ar[j], plane2);
        ui[j - j0] = Grp<64>::bcast(ai[j], plane2);
      }
#pragma unroll
    for (int j = j0; j < j0 + kBcastChunk; ++j)
      if (j < N) {
        ar[j] = fma(li, ui[j - j0], fma(-lr, ur[j - j0], ar[j]));
        ai[j] = fma(-li, ur[j - j0], fma(-lr, ui[j - j0], ai[j]));
        pin(ar[j]);
        pin(ai[j]);
      }
  }
  if constexpr (std::is_same<T, double>::value) __builtin_amdgcn_sched_barrier(0);
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void lu_real_step(const int k, T (&a)[R][N], int (&pos)[R], Perm<N>& perm,
                                             T (&rd)[R], int& info) {
  const int ln = Grp<G>::lane();
  int bkey = 0x7fffffff;
  T bv = T(-1);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool act = pos[q] >= k;
    const T v = fabs(a[q][k]);
    const int key = (pos[q] << 8) | Rows<N, G, R>::row(ln, q);
    const bool better = act && (v > bv || (v == bv && key < bkey));
    bv = better ? v : bv;
    bkey = better ? key : bkey;
  }
  group_argmax<G>(bv, bkey);
  const int prow = bkey & 0xff;
  const int ppos = bkey >> 8;
  const int plane = prow % G;
  const int pq = prow / G;
  perm.set(k, prow);
  T mine[R];
#pragma unroll
  for (int q = 0; q < R; ++q) mine[q] = a[q][k];
  const T piv = Grp<G>::bcast(sel<R>(mine, pq), plane);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool is_piv = Rows<N, G, R>::row(ln, q) == prow;
    pos[q] = is_piv ? k : (pos[q] == k ? ppos : pos[q]);  // LAPACK swaps rows k and ppos
  }
  const bool nz = piv != T(0);
  if (!nz && info == 0) info = k + 1;
  // LAPACK divides instead of scaling by the reciprocal when |pivot| < sfmin
  // (FP64 path only; the FP32 factors need no such care)
  const bool tiny = std::is_same<T, double>::value && fabs(piv) < min_normal<T>();
  const T rp = recip(piv);
  T l[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    rd[q] = (Rows<N, G, R>::row(ln, q) == prow) ? (nz ? rp : T(0)) : rd[q];
    const bool act = nz && pos[q] > k;
    const T lq = tiny ? a[q][k] / piv : a[q][k] * rp;
    l[q] = act ? lq : T(0);
    a[q][k] = act ? lq : a[q][k];
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j > k) {
      T m2[R];
#pragma unroll
      for (int q = 0; q < R; ++q) m2[q] = a[q][j];
      const T uj = Grp<G>::bcast(sel<R>(m2, pq), plane);
#pragma unroll
      for (int q = 0; q < R; ++q) a[q][j] = fma(-l[q], uj, a[q][j]);
    }
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void lu_real(T (&a)[R][N], int (&pos)[R], Perm<N>& perm,
                                        T (&rd)[R], int& info) {
  lu_init<N, G, R, T>(pos, rd, info);
#pragma unroll
  for (int k = 0; k < N; ++k) lu_real_step<N, G, R, T>(k, a, pos, perm, rd, info);
}

// ---- complex LU (zgetf2 semantics) -------------------------------------------
template <int N, int G, int R, class T>
__device__ __forceinline__ void lu_cplx_step(const int k, T (&ar)[R][N], T (&ai)[R][N], int (&pos)[R],
                                             Perm<N>& perm, T (&rdr)[R], T (&rdi)[R], int& info) {
  const int ln = Grp<G>::lane();
  int bkey = 0x7fffffff;
  T bv = T(-1);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool act = pos[q] >= k;
    const T v = fabs(ar[q][k]) + fabs(ai[q][k]);
    const int key = (pos[q] << 8) | Rows<N, G, R>::row(ln, q);
    const bool better = act && (v > bv || (v == bv && key < bkey));
    bv = better ? v : bv;
    bkey = better ? key : bkey;
  }
  group_argmax<G>(bv, bkey);
  const int prow = bkey & 0xff;
  const int ppos = bkey >> 8;
  const int plane = prow % G;
  const int pq = prow / G;
  perm.set(k, prow);
  T mr[R], mi[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { mr[q] = ar[q][k]; mi[q] = ai[q][k]; }
  const T pr_ = Grp<G>::bcast(sel<R>(mr, pq), plane);
  const T pi_ = Grp<G>::bcast(sel<R>(mi, pq), plane);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool is_piv = Rows<N, G, R>::row(ln, q) == prow;
    pos[q] = is_piv ? k : (pos[q] == k ? ppos : pos[q]);
  }
  const bool nz = (pr_ != T(0) || pi_ != T(0));
  if (!nz && info == 0) info = k + 1;
  T rr, ri;
  crecip(pr_, pi_, rr, ri);
  T lr[R], li[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool is_piv = Rows<N, G, R>::row(ln, q) == prow;
    rdr[q] = is_piv ? (nz ? rr : T(0)) : rdr[q];
    rdi[q] = is_piv ? (nz ? ri : T(0)) : rdi[q];
    const bool act = nz && pos[q] > k;
    const T xr = ar[q][k], xi = ai[q][k];
    const T vr = xr * rr - xi * ri;
    const T vi = xr * ri + xi * rr;
    lr[q] = act ? vr : T(0);
    li[q] = act ? vi : T(0);
    ar[q][k] = act ? vr : ar[q][k];
    ai[q][k] = act ? vi : ai[q][k];
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j > k) {
      T m2r[R], m2i[R];
#pragma unroll
      for (int q = 0; q < R; ++q) { m2r[q] = ar[q][j]; m2i[q] = ai[q][j]; }
      const T ur = Grp<G>::bcast(sel<R>(m2r, pq), plane);
      const T ui = Grp<G>::bcast(sel<R>(m2i, pq), plane);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        ar[q][j] = fma(-lr[q], ur, ar[q][j]);
        ar[q][j] = fma(li[q], ui, ar[q][j]);
        ai[q][j] = fma(-lr[q], ui, ai[q][j]);
        ai[q][j] = fma(-li[q], ur, ai[q][j]);
      }
    }
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void lu_cplx(T (&ar)[R][N], T (&ai)[R][N], int (&pos)[R],
                                        Perm<N>& perm, T (&rdr)[R], T (&rdi)[R],
                                        int& info) {
  lu_init<N, G, R, T>(pos, rdr, info);
#pragma unroll
  for (int q = 0; q < R; ++q) rdi[q] = T(0);
#pragma unroll
  for (int k = 0; k < N; ++k) lu_cplx_step<N, G, R, T>(k, ar, ai, pos, perm, rdr, rdi, info);
}

// The real and the complex LU of a 64-lane group, a row per lane, step by step
// together.
template <int N, class T>
__device__ __forceinline__ void wave_lu(T (&a)[1][N], int (&pos)[1], Perm<N>& perm, T (&rd)[1], int& info,
                                        T (&ar)[1][N], T (&ai)[1][N], int (&pos2)[1], Perm<N>& perm2, T (&rdr)[1],
                                        T (&rdi)[1], int& info2) {
  lu_init<N, 64, 1, T>(pos, rd, info);
  lu_init<N, 64, 1, T>(pos2, rdr, info2);
  rdi[0] = T(0);
  Perm<N> pm = {}, pm2 = {};  // built in scalar registers
  int inf = 0, inf2 = 0;
#pragma unroll
  for (int k = 0; k < N; ++k)
    wave_lu_step<N, T>(k, a[0], pos[0], pm, rd[0], inf, ar[0], ai[0], pos2[0], pm2, rdr[0], rdi[0], inf2);
  perm = pm;
  perm2 = pm2;
  info = inf;
  info2 = inf2;
}

// ---- triangular solves (dgetrs / zgetrs, nrhs = 1) ---------------------------
// A solve's view of the row positions and of the pivot rows.  The rows that do
// not take part in a step keep their right-hand side by a select on the
// result; both the positions and (64-lane groups) the pivot rows, read into
// scalar registers, are opaque to the compiler, so that no select, compare or
// table entry looks invariant in the Newton loop: hoisted out of it, the
// masked copies of all three factors alone needed as many registers as the
// factors again, and every solve read them back from scratch.
template <int N, int G, int R>
struct SolveView {
  int pos[R];
  Perm<N> perm;
  __device__ __forceinline__ SolveView(const int (&p)[R], const Perm<N>& pm) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      pos[q] = p[q];
      __asm__ volatile("" : "+v"(pos[q]));
    }
#pragma unroll
    for (int i = 0; i < (N + 3) / 4; ++i) {
      if constexpr (G == 64) {
        perm.w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)pm.w[i]);
        __asm__ volatile("" : "+s"(perm.w[i]));
      } else {
        perm.w[i] = pm.w[i];
      }
    }
  }
};

// b[q] is the right-hand side of row r = row(ln, q); on return it holds
// solution component r.  Forward then backward column-oriented substitution in
// pivot order, as reference BLAS dtrsm does it; rows outside the current
// step's range take a zero coefficient.
template <int N, int G, int R, class T>
__device__ __forceinline__ void fwd_real_step(const int k, const T (&a)[R][N], const int (&pos)[R],
                                              const Perm<N>& perm, T (&b)[R]) {
  const int prow = perm.get(k);
  const T yk = Grp<G>::bcast(sel<R>(b, prow / G), prow % G);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const T v = fma(-a[q][k], yk, b[q]);
    b[q] = pos[q] > k ? v : b[q];
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void bwd_real_step(const int k, const T (&a)[R][N], const int (&pos)[R],
                                              const Perm<N>& perm, const T (&rd)[R], T (&b)[R], T (&x)[R]) {
  const int ln = Grp<G>::lane();
  const int prow = perm.get(k);
  const int pq = prow / G;
  const T xk = Grp<G>::bcast(sel<R>(b, pq) * sel<R>(rd, pq), prow % G);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const T v = fma(-a[q][k], xk, b[q]);
    b[q] = (unsigned)pos[q] < (unsigned)k ? v : b[q];  // (pos = -1: padding rows)
    x[q] = (Rows<N, G, R>::row(ln, q) == k) ? xk : x[q];
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void solve_real(const T (&a)[R][N], const int (&pos)[R],
                                           const Perm<N>& perm, const T (&rd)[R],
                                           T (&b)[R]) {
  const SolveView<N, G, R> v(pos, perm);
#pragma unroll
  for (int k = 0; k < N; ++k) fwd_real_step<N, G, R, T>(k, a, v.pos, v.perm, b);
  T x[R];
#pragma unroll
  for (int q = 0; q < R; ++q) x[q] = T(0);
#pragma unroll
  for (int k = N - 1; k >= 0; --k) bwd_real_step<N, G, R, T>(k, a, v.pos, v.perm, rd, b, x);
#pragma unroll
  for (int q = 0; q < R; ++q) b[q] = x[q];
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void fwd_cplx_step(const int k, const T (&ar)[R][N], const T (&ai)[R][N],
                                              const int (&pos)[R], const Perm<N>& perm, T (&br)[R], T (&bi)[R]) {
  const int prow = perm.get(k);
  const int pl = prow % G, pq = prow / G;
  const T yr = Grp<G>::bcast(sel<R>(br, pq), pl);
  const T yi = Grp<G>::bcast(sel<R>(bi, pq), pl);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool act = pos[q] > k;
    const T lr = ar[q][k], li = ai[q][k];
    const T vr = fma(li, yi, fma(-lr, yr, br[q]));
    const T vi = fma(-li, yr, fma(-lr, yi, bi[q]));
    br[q] = act ? vr : br[q];
    bi[q] = act ? vi : bi[q];
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void bwd_cplx_step(const int k, const T (&ar)[R][N], const T (&ai)[R][N],
                                              const int (&pos)[R], const Perm<N>& perm, const T (&rdr)[R],
                                              const T (&rdi)[R], T (&br)[R], T (&bi)[R], T (&xr)[R], T (&xi)[R]) {
  const int ln = Grp<G>::lane();
  const int prow = perm.get(k);
  const int pl = prow % G, pq = prow / G;
  const T vr = sel<R>(br, pq), vi = sel<R>(bi, pq);
  const T dr = sel<R>(rdr, pq), di = sel<R>(rdi, pq);
  const T kr = Grp<G>::bcast(vr * dr - vi * di, pl);
  const T ki = Grp<G>::bcast(vr * di + vi * dr, pl);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool act = (unsigned)pos[q] < (unsigned)k;
    const T ur = ar[q][k], ui = ai[q][k];
    const T vr2 = fma(ui, ki, fma(-ur, kr, br[q]));
    const T vi2 = fma(-ui, kr, fma(-ur, ki, bi[q]));
    br[q] = act ? vr2 : br[q];
    bi[q] = act ? vi2 : bi[q];
    const bool mine = Rows<N, G, R>::row(ln, q) == k;
    xr[q] = mine ? kr : xr[q];
    xi[q] = mine ? ki : xi[q];
  }
}

template <int N, int G, int R, class T>
__device__ __forceinline__ void solve_cplx(const T (&ar)[R][N], const T (&ai)[R][N],
                                           const int (&pos)[R], const Perm<N>& perm,
                                           const T (&rdr)[R], const T (&rdi)[R],
                                           T (&br)[R], T (&bi)[R]) {
  const SolveView<N, G, R> v(pos, perm);
#pragma unroll
  for (int k = 0; k < N; ++k) fwd_cplx_step<N, G, R, T>(k, ar, ai, v.pos, v.perm, br, bi);
  T xr[R], xi[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { xr[q] = T(0); xi[q] = T(0); }
#pragma unroll
  for (int k = N - 1; k >= 0; --k) bwd_cplx_step<N, G, R, T>(k, ar, ai, v.pos, v.perm, rdr, rdi, br, bi, xr, xi);
#pragma unroll
  for (int q = 0; q < R; ++q) { br[q] = xr[q]; bi[q] = xi[q]; }
}

// Orders LDS traffic between lanes of one wavefront (a group never spans
// waves): LDS operations of a wave complete in issue order, so a compiler
// barrier plus an LDS-counter wait suffices; no global-memory wait is implied.
__device__ __forceinline__ void group_lds_sync() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt/expcnt untouched
  __builtin_amdgcn_wave_barrier();
  __asm__ volatile("" ::: "memory");
}

// ---- compile-time-lane primitives -------------------------------------------
// Loops whose index must be a constant expression (a DPP control or a readlane
// lane) are written with static_for.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// Broadcast the value held by lane K of each lane group to the whole group.
// G = 16: DPP row_newbcast (one VALU move per dword, no LDS round trip);
// G = 64: readlane into SGPRs; other widths fall back to ds_bpermute.
template <int G, int K>
__device__ __forceinline__ int bcast_k_i(int v) {
  if constexpr (G == 1) {
    return v;
  } else if constexpr (G == 16) {
    return __builtin_amdgcn_mov_dpp(v, 0x150 + K, 0xf, 0xf, false);
  } else if constexpr (G == 64) {
    return __builtin_amdgcn_readlane(v, K);
  } else {
    return __shfl(v, K, G);
  }
}
template <int G, int K>
__device__ __forceinline__ float bcast_k(float v) {
  return __int_as_float(bcast_k_i<G, K>(__float_as_int(v)));
}
template <int G, int K>
__device__ __forceinline__ double bcast_k(double v) {
  if constexpr (G == 1) {
    return v;
  } else {
    const int lo = bcast_k_i<G, K>(__double2loint(v));
    const int hi = bcast_k_i<G, K>(__double2hiint(v));
    return __hiloint2double(hi, lo);
  }
}

// ---- LU of 16-lane groups (N <= 16, a row per lane; four systems a wavefront) --
// dgetf2 / zgetf2 semantics like the row LU above.  The pivot search exchanges
// the leading 32 bits of the magnitudes inside the DPP row of the group (four
// v_max_u32 with the exchange folded in) and reads the winner from the group's
// 16 bits of one compare mask; rows that agree in those bits, which is rare, go
// through the full (value, position) search.  The pivot row is in a lane that
// differs from group to group, so its entries are gathered (ds_bpermute, all
// columns of a step in flight behind the reciprocal).  At the end the rows move
// to the lanes of their LAPACK positions, so that the solves broadcast from
// compile-time lanes on the VALU.
//
// Bound by issue and the gathers' latency at two waves per SIMD.  It replaced a
// lane-per-column LU (pivot search down a lane's registers, interchanges as
// selects in every lane) of 58k cycles per FP64 pair at order 14, and in FP32
// a row LU with gathered solves; measured on 262144 14-state conditions of two
// steps: FP64 30.0 -> 17.3 ms, 30011 conditions of four steps with FP32 factors
// 4.26 -> 3.40 ms (with the Jacobian's batches).
__device__ __forceinline__ int bperm(int addr, int v) { return __builtin_amdgcn_ds_bpermute(addr, v); }
__device__ __forceinline__ float bperm(int addr, float v) { return __int_as_float(bperm(addr, __float_as_int(v))); }
__device__ __forceinline__ double bperm(int addr, double v) {
  const int lo = bperm(addr, __double2loint(v)), hi = bperm(addr, __double2hiint(v));
  return __hiloint2double(hi, lo);
}

// Pivot row of a step: the lane of the group (first maximum of the magnitudes v
// over the active rows in LAPACK's order pos), or 0xff if no active row holds a
// comparable value.
template <class T>
__device__ __forceinline__ int row16_pivot(T v, int pos, bool act) {
  const unsigned key = act && v == v ? mag_hi(v) + 1u : 0u;  // 0: no candidate
  unsigned m = dpp_max_u<kDppXor1>(key);
  m = dpp_max_u<kDppXor2>(m);
  m = dpp_max_u<kDppHalfMirror>(m);
  m = dpp_max_u<kDppMirror>(m);
  const unsigned long long all = __builtin_amdgcn_ballot_w64(key == m);
  const int lane = (int)__lane_id();
  const unsigned half = (lane & 32) ? (unsigned)(all >> 32) : (unsigned)all;
  const unsigned cand = (half >> (lane & 16)) & 0xffffu;
  int prow = __builtin_ctz(cand | 0x10000u);
  if (__builtin_expect((cand & (cand - 1)) != 0, 0)) {
    T bv = act && v == v ? v : T(-1);
    int bkey = act && v == v ? ((pos << 8) | (lane & 15)) : 0x7fffffff;
    group_argmax<16>(bv, bkey);
    prow = bkey & 0xff;
  }
  return prow;
}

// Rows to the lanes of their positions: src = the row (lane) whose position is
// this lane's index.
__device__ __forceinline__ int row16_source(int pos) {
  const int lane = (int)__lane_id(), base = lane & 48;
  const int to = pos >= 0 ? (pos & 15) : (lane & 15);
  return __builtin_amdgcn_ds_permute((base | to) << 2, lane & 15) & 15;
}

template <int N, class T>
__device__ __forceinline__ void row16_lu_real(T (&a)[N], int& src, T& rd, int& info) {
  static_assert(N <= 16, "a 16-lane group holds at most 16 rows");
  const int ln = Grp<16>::lane(), base = (int)__lane_id() & 48;
  int pos = ln < N ? ln : -1;
  rd = T(0);
  info = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int prow = row16_pivot(fabs(a[k]), pos, pos >= k);
    const int from = (base | (prow & 15)) << 2;
    const int ppos = prow == 0xff ? 0x7fffff : bperm(from, pos);
    const T piv = bperm(from, a[k]);
    T u[N];
#pragma unroll
    for (int j = k + 1; j < N; ++j) u[j] = bperm(from, a[j]);
    const bool is_piv = ln == prow;
    pos = is_piv ? k : (pos == k ? ppos : pos);
    pin(pos);
    const bool nz = piv != T(0);
    info = !nz && info == 0 ? k + 1 : info;
    pin(info);
    const T rp = recip(piv);
    T lq = a[k] * rp;
    if constexpr (std::is_same<T, double>::value)
      if (__builtin_expect(fabs(piv) < min_normal<T>(), 0)) lq = a[k] / piv;
    rd = is_piv ? (nz ? rp : T(0)) : rd;
    pin(rd);
    const bool act = nz && pos > k;
    a[k] = act ? lq : a[k];
    T l = act ? -lq : T(-0.0);
    pin(a[k]);
    pin(l);
#pragma unroll
    for (int j = k + 1; j < N; ++j) {
      a[j] = fma(l, u[j], a[j]);
      pin(a[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  src = row16_source(pos);
  const int from = (base | src) << 2;
#pragma unroll
  for (int j = 0; j < N; ++j) a[j] = bperm(from, a[j]);
  rd = bperm(from, rd);
}

template <int N, class T>
__device__ __forceinline__ void row16_lu_cplx(T (&ar)[N], T (&ai)[N], int& src, T& rdr, T& rdi, int& info) {
  static_assert(N <= 16, "a 16-lane group holds at most 16 rows");
  const int ln = Grp<16>::lane(), base = (int)__lane_id() & 48;
  int pos = ln < N ? ln : -1;
  rdr = rdi = T(0);
  info = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int prow = row16_pivot(fabs(ar[k]) + fabs(ai[k]), pos, pos >= k);
    const int from = (base | (prow & 15)) << 2;
    const int ppos = prow == 0xff ? 0x7fffff : bperm(from, pos);
    const T pr_ = bperm(from, ar[k]), pi_ = bperm(from, ai[k]);
    T ur[N], ui[N];
#pragma unroll
    for (int j = k + 1; j < N; ++j) {
      ur[j] = bperm(from, ar[j]);
      ui[j] = bperm(from, ai[j]);
    }
    const bool is_piv = ln == prow;
    pos = is_piv ? k : (pos == k ? ppos : pos);
    pin(pos);
    const bool nz = pr_ != T(0) || pi_ != T(0);
    info = !nz && info == 0 ? k + 1 : info;
    pin(info);
    T rr, ri;
    crecip(pr_, pi_, rr, ri);
    rdr = is_piv ? (nz ? rr : T(0)) : rdr;
    rdi = is_piv ? (nz ? ri : T(0)) : rdi;
    pin(rdr);
    pin(rdi);
    const bool act = nz && pos > k;
    const T xr = ar[k], xi = ai[k];
    const T vr = xr * rr - xi * ri;
    const T vi = xr * ri + xi * rr;
    ar[k] = act ? vr : xr;
    ai[k] = act ? vi : xi;
    T lr = act ? vr : T(0), li = act ? vi : T(0);
    pin(ar[k]);
    pin(ai[k]);
    pin(lr);
    pin(li);
#pragma unroll
    for (int j = k + 1; j < N; ++j) {
      ar[j] = fma(li, ui[j], fma(-lr, ur[j], ar[j]));
      ai[j] = fma(-li, ur[j], fma(-lr, ui[j], ai[j]));
      pin(ar[j]);
      pin(ai[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  src = row16_source(pos);
  const int from = (base | src) << 2;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    ar[j] = bperm(from, ar[j]);
    ai[j] = bperm(from, ai[j]);
  }
  rdr = bperm(from, rdr);
  rdi = bperm(from, rdi);
}

// ---- row-layout solves for the explicit-interchange factors ----------------
// 16-lane groups: lane i holds row i of L\U (LAPACK order) and src = the original
// row whose equation sits in position i; b[] is the right-hand side of the lane's own
// (original) equation.  Pivot rows are at compile-time lanes, so every
// broadcast comes from a fixed lane.  On return b holds solution component i
// in lane i.
// (The triangles are masked by compile-time steps against the lane, so the
// coefficients are taken as they are and the rows outside a step keep x by a
// select: see SolveView.)
template <int N, int G, class T>
__device__ __forceinline__ void rsolve_real(const T (&a)[N], int src, T rdiag, T& b) {
  int ln = Grp<G>::lane();
  pin(ln);
  T x = __shfl(b, src, G);  // (P b)_i
  static_for<0, N>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    const T v = fma(-a[k], bcast_k<G, k>(x), x);
    x = ln > k && ln < N ? v : x;
  });
  static_for<0, N>([&](auto kc) {
    constexpr int k = N - 1 - decltype(kc)::value;
    const T xk = bcast_k<G, k>(x * rdiag);
    const T v = fma(-a[k], xk, x);
    x = ln < k ? v : (ln == k ? xk : x);
  });
  b = (ln < N) ? x : T(0);
}

template <int N, int G, class T>
__device__ __forceinline__ void rsolve_cplx(const T (&ar)[N], const T (&ai)[N], int src, T rdr, T rdi, T& br, T& bi) {
  int ln = Grp<G>::lane();
  pin(ln);
  T xr = __shfl(br, src, G), xi = __shfl(bi, src, G);
  static_for<0, N>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    const T yr = bcast_k<G, k>(xr), yi = bcast_k<G, k>(xi);
    const bool act = ln > k && ln < N;
    const T vr = fma(ai[k], yi, fma(-ar[k], yr, xr));
    const T vi = fma(-ai[k], yr, fma(-ar[k], yi, xi));
    xr = act ? vr : xr;
    xi = act ? vi : xi;
  });
  static_for<0, N>([&](auto kc) {
    constexpr int k = N - 1 - decltype(kc)::value;
    const T kr = bcast_k<G, k>(xr * rdr - xi * rdi);
    const T ki = bcast_k<G, k>(xr * rdi + xi * rdr);
    const T vr = fma(ai[k], ki, fma(-ar[k], kr, xr));
    const T vi = fma(-ai[k], kr, fma(-ar[k], ki, xi));
    xr = ln < k ? vr : (ln == k ? kr : xr);
    xi = ln < k ? vi : (ln == k ? ki : xi);
  });
  br = (ln < N) ? xr : T(0);
  bi = (ln < N) ? xi : T(0);
}

// ---- the integrator ----------------------------------------------------------
// Mech provides:
//   static constexpr int N;
//   struct Ctx;  (per-group context: LDS pointers, tables)
//   template <int G, int R> dydt(Ctx&, t, pr, const double (&y)[R], double (&f)[R])
//   static constexpr bool kJacInLds;  double* Ctx::jac  (N*N doubles when true)
//   kJacInLds:  template <int G, int R> jacob(Ctx&, t, pr, const double (&y)[R])
//               writing rows ctx.jac[r*N + j] = d f_r / d y_j
//   otherwise:  template <int G, int R> jacob(Ctx&, t, pr, const double (&y)[R], double (&J)[R][N])
// When kJacInLds is set the Jacobian lives in the group's LDS (it is only read
// when the iteration matrices are rebuilt), which keeps N*R doubles per lane
// out of the register file.
//
// The reference's integrate() (radau2a.c:520-736) is a loop over step
// attempts.  Here it is a resumable state machine: begin() is the prologue
// (:521-564) and attempt() runs one pass of the loop body (:566-734) and
// reports whether the interval is finished, so a persistent kernel can
// interleave step attempts of many conditions and refill a lane group with a
// new condition or a new global step as soon as its current one ends.
enum : int { RADAU_CONTINUE = -1 };

}  // namespace acc
#include "lu_mem.hpp"
namespace acc {

// The step controller's powers.  pow() itself is ~250 instructions, called two to
// four times per attempt with all of the integrator's state live (a third of a
// van der Pol attempt); the exponents that occur every time are fixed, so they
// take Newton's iteration on the root from a hardware FP32 start (relative error
// 1e-6, squared twice): 15 instructions, inline.  Largest error over the ranges
// below, 1e7 arguments each against 80-bit arithmetic, in units of 2^-53:
// inv_root4 1.60 (pow 1.98), pow_0p8 2.24, pow_int 1.99.  With the norms' shared
// root and the quotients by H and by constants from one reciprocal (quot):
// 262144 oscillators of five steps 0.82 -> 0.58 ms, 262144 14-state conditions of
// two steps 17.3 -> 15.7 ms (FP64), 65536 54-state ones with FP32 factors
// 162.1 -> 157.6 ms.
//
// x^(-1/4), x > 0; arguments above 1e38 count as 1e38 (the controller's factors
// are clamped long before).
__device__ __forceinline__ double inv_root4(double x) {
  x = fmin(x, 1e38);
  double y = (double)__builtin_amdgcn_rsqf(__builtin_amdgcn_sqrtf((float)x));
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // y += y (1 - x y^4) / 4
    const double y2 = y * y;
    y = fma(y, 0.25 * fma(-(x * y2), y2, 1.0), y);
  }
  return y;
}
// x^0.8 = x x^(-1/5), 1e-16 <= x <= 1e3 (the Newton rate).
__device__ __forceinline__ double pow_0p8(double x) {
  double y = (double)__builtin_amdgcn_exp2f(-0.2f * __builtin_amdgcn_logf((float)x));
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // y += y (1 - x y^5) / 5
    const double y2 = y * y;
    y = fma(y, 0.2 * fma(-(x * y), y2 * y2, 1.0), y);
  }
  return x * y;
}
// x^n, 0 <= n <= 7, the products' rounding errors carried along.
__device__ __forceinline__ double pow_int(double x, int n) {
  const double x2 = x * x, e2 = fma(x, x, -x2);
  const double x4 = x2 * x2, e4 = fma(x2, x2, -x4) + 2.0 * x2 * e2;
  double p = (n & 1) ? x : 1.0, e = 0.0;
  const double p2 = p * x2, f2 = fma(p, x2, -p2) + p * e2;
  p = (n & 2) ? p2 : p;
  e = (n & 2) ? f2 : e;
  const double p4 = p * x4, f4 = fma(p, x4, -p4) + (p * e4 + e * x4);
  return (n & 4) ? p4 + f4 : p + e;
}
// x / d from the reciprocal id = 1 / d: the product corrected by its residual,
// which gives the quotient's rounding (all but exceptional last bits) in three
// instructions instead of a division's eleven.
__device__ __forceinline__ double quot(double x, double d, double id) {
  const double q = x * id;
  return fma(fma(-q, d, x), id, q);
}
// The step factor of a failing Newton iteration has an exponent that depends on
// the iteration: pow as a real call, so that its temporaries stay out of the
// integrator's register allocation (inlined, they spilled around the site).
__device__ __attribute__((noinline)) inline double step_pow(double x, double y) { return pow(x, y); }

template <class Mech, int G, int R, class MT = double>
struct Radau {
  static constexpr int N = Mech::N;
  using RW = Rows<N, G, R>;
  using Ctx = typename Mech::Ctx;
  // Matrix scalar type: double, or float for the mixed-precision method
  // (iteration-matrix factorizations and Newton solves in FP32; residuals,
  // error estimate, step control and state in FP64).
  static constexpr bool kMixed = std::is_same<MT, float>::value;
  static_assert(kMixed || std::is_same<MT, double>::value, "matrix type must be float or double");
  // 16-lane groups: the row LU that ends with every row in the lane of its
  // position (row16_lu_*), and solves with compile-time broadcast lanes.
  static constexpr bool kRow16 = G == 16 && R == 1;
  // Systems above 64 states: a wavefront per condition (R rows per lane), the
  // factorizations in a per-wave global workspace (MemLU: blocked LU with
  // MFMA trailing updates) instead of registers.
  static constexpr bool kMemLU = N > 64;
  static_assert(!kMemLU || (G == 64 && Mech::kJacInLds), "large systems: one wavefront per condition");
  using MLU = MemLU<(kMemLU ? N : 80), (kMemLU ? R : 2), MT>;
  static constexpr int NF = kMemLU ? 1 : N;  // register-resident factor columns
  static constexpr int kRowMaxUnroll = kMemLU ? 4 : N;

  // per-interval controller state (group-uniform)
  double t, t_end, H, Hold, Hacc, ErrOld, NewtonRate;
  int Nconsecutive, Nsteps;
  bool Reject, FirstStep, SkipJac, SkipLU;
  // row-owned vectors
  double y[R], sc[R], y0[R], F0[R], Z1[R], Z2[R], Z3[R];
  double CONT0[R], CONT1[R], CONT2[R];
  // factorizations (registers; for kMemLU in the workspace at ws)
  MT E1[R][NF], E2r[R][NF], E2i[R][NF];
  MT* ws = nullptr;
  int pos1[R], pos2[R];
  // mixed precision: each matrix is scaled on both sides by powers of two
  // (exact), D_r M D_c with D_r = 2^-ex, D_c = 2^-cx, before rounding to FP32:
  // kEquilSweeps sweeps of Ruiz equilibration (row, then column maxima halved
  // in exponent towards 1), then every row normalised so its largest entry
  // lies in [0.5, 1).  Jacobian entries of stiff kinetics span tens of orders
  // of magnitude across rows and columns and reach beyond the FP32 range; with
  // rows scaled alone the iteration matrices kept condition numbers of 1e6 -
  // 1e9 (54 states) and 1e9 - 1e13 (112 states), beyond what FP32 factors
  // resolve; three sweeps bring them to 1e2 - 1e3.  The scaled system's
  // solution is D_c^-1 x, so the solves scale back by 2^-cx.
  // Up to 64 states (factors in registers) the column exponents are chosen
  // once per Jacobian instead -- half the binary exponent of the diagonal of
  // gamma/H - J at that evaluation -- and the parked Jacobian is stored
  // column-scaled (park_column_scaling), so forming E1, E2 needs no
  // per-column broadcasts (which cost the 54-state launch 16 - 55 %); only
  // the row pass runs per factorization.  With that scaling the 131072-
  // condition 54-state window ends every condition within 10 tolerance units
  // of FP64 (max 7.3; rows alone: 144 beyond, max 201).
  static constexpr int kEquilSweeps = 3;
  // row exponents of the rows this lane holds, and column exponents of the
  // columns with the same indices (E1, E2).  Register path: one column scale
  // for both matrices (cx1), and both row exponents packed into ex1 (16 bits
  // each: fewer live registers in a kernel that spills).
  int ex1[R], ex2[kMemLU ? R : 1];
  int cx1[R], cx2[kMemLU ? R : 1];
  __device__ __forceinline__ int row_exp1(int q) const { return kMemLU ? ex1[q] : (int)(short)(ex1[q] & 0xffff); }
  __device__ __forceinline__ int row_exp2(int q) const { return kMemLU ? ex2[q] : ex1[q] >> 16; }
  MT rd1[R], rd2r[R], rd2i[R];
  Perm<N> perm1, perm2;
  int src1, src2;  // 16-lane groups: original equation of this lane's row
  double A[R][N];  // Jacobian (only live across attempts when !Mech::kJacInLds)
  // predicted Newton start of the current global step's first step; dropped
  // (zero start, the reference's rule) after any rejection of that step
  // kept in the group's LDS slice (zs[s*G*R + q*G + lane], s = stage), not in
  // registers: it is read once, at the start of the first step
  double* zs = nullptr;
  bool UseStart;
  // set when a predicted start was discarded (by the first-iteration test or
  // a Newton failure) or needed three or more Newton iterations; the caller
  // stops predicting for this condition
  bool StartFailed;

  __device__ __forceinline__ void set_start(const double (&z1)[R], const double (&z2)[R], const double (&z3)[R]) {
    const int ln = Grp<G>::lane();
#pragma unroll
    for (int q = 0; q < R; ++q) {
      zs[q * G + ln] = z1[q];
      zs[(R + q) * G + ln] = z2[q];
      zs[(2 * R + q) * G + ln] = z3[q];
    }
    UseStart = true;
  }

  __device__ __forceinline__ MT* wE1() const { return ws; }
  __device__ __forceinline__ MT* wE2r() const { return ws + MLU::kMat; }
  __device__ __forceinline__ MT* wE2i() const { return ws + 2 * MLU::kMat; }
  __device__ __forceinline__ int* wperm1() const { return MLU::perm1(ws); }
  __device__ __forceinline__ int* wperm2() const { return MLU::perm2(ws); }

  __device__ __forceinline__ void solve1(double (&b)[R]) const {
    if constexpr (kMemLU) {
      MT bb[R];
#pragma unroll
      for (int q = 0; q < R; ++q) bb[q] = kMixed ? (MT)ldexp(b[q], -ex1[q]) : (MT)b[q];
      MLU::solve_real(wE1(), wperm1(), bb);
#pragma unroll
      for (int q = 0; q < R; ++q) b[q] = kMixed ? ldexp((double)bb[q], -cx1[q]) : (double)bb[q];
    } else if constexpr (kRow16) {
      MT x = kMixed ? (MT)ldexp(b[0], -row_exp1(0)) : (MT)b[0];
      rsolve_real<N, G, MT>(E1[0], src1, rd1[0], x);
      b[0] = kMixed ? ldexp((double)x, -cx1[0]) : (double)x;
    } else if constexpr (!kMixed) {
      solve_real<N, G, R, double>(E1, pos1, perm1, rd1, b);
    } else {
      MT bb[R];
#pragma unroll
      for (int q = 0; q < R; ++q) bb[q] = (MT)ldexp(b[q], -row_exp1(q));
      solve_real<N, G, R, MT>(E1, pos1, perm1, rd1, bb);
#pragma unroll
      for (int q = 0; q < R; ++q) b[q] = ldexp((double)bb[q], -cx1[q]);
    }
  }
  __device__ __forceinline__ void solve2(double (&br)[R], double (&bi)[R]) const {
    if constexpr (kMemLU) {
      MT xr[R], xi[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        xr[q] = kMixed ? (MT)ldexp(br[q], -ex2[q]) : (MT)br[q];
        xi[q] = kMixed ? (MT)ldexp(bi[q], -ex2[q]) : (MT)bi[q];
      }
      MLU::solve_cplx(wE2r(), wE2i(), wperm2(), xr, xi);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        br[q] = kMixed ? ldexp((double)xr[q], -cx2[q]) : (double)xr[q];
        bi[q] = kMixed ? ldexp((double)xi[q], -cx2[q]) : (double)xi[q];
      }
    } else if constexpr (kRow16) {
      MT xr = kMixed ? (MT)ldexp(br[0], -row_exp2(0)) : (MT)br[0];
      MT xi = kMixed ? (MT)ldexp(bi[0], -row_exp2(0)) : (MT)bi[0];
      rsolve_cplx<N, G, MT>(E2r[0], E2i[0], src2, rd2r[0], rd2i[0], xr, xi);
      br[0] = kMixed ? ldexp((double)xr, -cx1[0]) : (double)xr;
      bi[0] = kMixed ? ldexp((double)xi, -cx1[0]) : (double)xi;
    } else if constexpr (!kMixed) {
      solve_cplx<N, G, R, double>(E2r, E2i, pos2, perm2, rd2r, rd2i, br, bi);
    } else {
      MT xr[R], xi[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        xr[q] = (MT)ldexp(br[q], -row_exp2(q));
        xi[q] = (MT)ldexp(bi[q], -row_exp2(q));
      }
      solve_cplx<N, G, R, MT>(E2r, E2i, pos2, perm2, rd2r, rd2i, xr, xi);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        br[q] = ldexp((double)xr[q], -cx1[q]);
        bi[q] = ldexp((double)xi[q], -cx1[q]);
      }
    }
  }

  // Entry (row(ln, q), j) of the parked Jacobian, 0 for rows beyond N.  In
  // global memory (the column-major layout of the large systems) the load is
  // unconditional, of an in-bounds row, followed by a select: a masked load
  // per entry makes the compiler keep every entry's address live.
  __device__ __forceinline__ static double jac_entry(const Ctx& ctx, int ln, int q, int j) {
    if constexpr (JacColMajor<Mech>::value) {
      const double v = ctx.jac[jidx<Mech>(RW::valid(ln, q) ? RW::row(ln, q) : 0, j)];
      return RW::valid(ln, q) ? v : 0.0;
    } else {
      return RW::valid(ln, q) ? ctx.jac[jidx<Mech>(RW::row(ln, q), j)] : 0.0;
    }
  }

  // Error-estimate solve.  FP64 factors: one solve.  FP32 factors: one solve
  // plus one step of iterative refinement against the FP64 matrix
  // gamma/H - J (J = the Jacobian the factors were built from), so the
  // estimate keeps FP64 accuracy whenever cond(E1) * 2^-24 << 1.
  __device__ __forceinline__ void solve1_es(Ctx& ctx, double (&b)[R]) const {
    if constexpr (!kMixed) {
      solve1(b);
    } else {
      const int ln = Grp<G>::lane();
      double x[R];
#pragma unroll
      for (int q = 0; q < R; ++q) x[q] = b[q];
      solve1(x);
      if constexpr (Mech::kJacInLds) group_lds_sync();
      const double g1 = rkGamma / H;
      double r[R];
#pragma unroll
      for (int q = 0; q < R; ++q) r[q] = b[q] - g1 * x[q];
      if constexpr (kMemLU) {
        // a rolled loop: unrolled over 112 columns the compiler hoists every
        // Jacobian load of both rows and spills them
#pragma unroll 4
        for (int j = 0; j < N; ++j) {
          const double xj = Grp<G>::bcast(sel<R>(x, j / G), j % G);
#pragma unroll
          for (int q = 0; q < R; ++q) {
            const double Jrj = jac_entry(ctx, ln, q, j);
            r[q] = fma(Jrj, xj, r[q]);
          }
        }
      } else {
        // J x = J' (D_c^-1 x): the parked Jacobian is column-scaled
        double xs[R];
#pragma unroll
        for (int q = 0; q < R; ++q) xs[q] = ldexp(x[q], cx1[q]);
        static_for<0, N>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          const double xj = bcast_k<G, j % G>(xs[j / G]);
#pragma unroll
          for (int q = 0; q < R; ++q) {
            double Jrj;
            if constexpr (Mech::kJacInLds) Jrj = jac_entry(ctx, ln, q, j);
            else Jrj = A[q][j];
            r[q] = fma(Jrj, xj, r[q]);
          }
        });
      }
#pragma unroll
      for (int q = 0; q < R; ++q) r[q] = RW::valid(ln, q) ? r[q] : 0.0;
      solve1(r);
#pragma unroll
      for (int q = 0; q < R; ++q) b[q] = x[q] + r[q];
    }
  }

  // Register path, mixed precision: the parked Jacobian J' = J D_c, with
  // D_c = 2^-cx and cx_j half the binary exponent of |gamma/H - J_jj| now;
  // each lane scales its own rows.  Exact (powers of two), and undone where J
  // itself is needed (J x = J' (D_c^-1 x) in the error estimate's refinement).
  __device__ __forceinline__ void park_column_scaling(Ctx& ctx) {
    const int ln = Grp<G>::lane();
    const double g1 = rkGamma / H;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = RW::row(ln, q);
      double djj;
      if constexpr (Mech::kJacInLds) djj = jac_entry(ctx, ln, q, RW::valid(ln, q) ? r : 0);
      else djj = A[q][RW::valid(ln, q) ? r : 0];
      const double m = fabs(g1 - djj);
      int e = 0;
      if (m > 0.0) frexp(m, &e);
      cx1[q] = RW::valid(ln, q) ? e / 2 : 0;
    }
    if constexpr (Mech::kJacInLds) {
#pragma unroll 4
      for (int j = 0; j < N; ++j) {
        const int cj = col_exp(cx1, j);
#pragma unroll
        for (int q = 0; q < R; ++q)
          if (RW::valid(ln, q)) {
            double& v = ctx.jac[jidx<Mech>(RW::row(ln, q), j)];
            v = ldexp(v, -cj);
          }
      }
      group_lds_sync();
    } else {
      static_for<0, N>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const int cj = bcast_k_i<G, j % G>(cx1[j / G]);
#pragma unroll
        for (int q = 0; q < R; ++q) A[q][j] = ldexp(A[q][j], -cj);
      });
    }
  }

  // Register path, mixed precision: row exponents of the column-scaled
  // matrix diag(dr + i di) D_c - J' (row r's diagonal scaled by its own
  // column's 2^-cx).
  template <class JA>
  __device__ __forceinline__ void row_exponents(JA&& jac_at, double dr, double di, int (&ex)[R]) const {
    const int ln = Grp<G>::lane();
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = RW::row(ln, q);
      const double sr = ldexp(dr, -cx1[q]), si = ldexp(di, -cx1[q]);
      double mx = 0.0;
#pragma unroll kRowMaxUnroll
      for (int j = 0; j < N; ++j) {
        const bool d = (j == r);
        mx = fmax(mx, fabs(-jac_at(q, r, j) + (d ? sr : 0.0)) + (d ? si : 0.0));
      }
      int e = 0;
      if (mx > 0.0) frexp(mx, &e);
      ex[q] = e;
    }
  }

  // Column exponent c_j (held by the lane of row j), runtime j.
  __device__ __forceinline__ static int col_exp(const int (&cx)[R], int j) {
    return Grp<G>::bcast_i(sel<R>(cx, j / G), j % G);
  }

  // Power-of-two two-sided scaling of M = diag(dr + i di) - J (magnitudes
  // |Re| + |Im|), as described at ex1 / cx1: column exponents cx of the
  // columns with this lane's row indices, row exponents ex of its rows.  The
  // sweeps work on binary exponents only (integer maxima of exponent
  // differences), so no intermediate can overflow; the final row exponents
  // make every scaled entry smaller than 1.
  template <class JA>
  __device__ __forceinline__ void equilibrate(JA&& jac_at, double dr, double di, int (&ex)[R], int (&cx)[R]) const {
    const int ln = Grp<G>::lane();
    constexpr int kZero = -100000;  // exponent of a zero entry
    auto eps = [&](int q, int j) -> int {
      const int r = RW::row(ln, q);
      const bool d = j == r;
      const double m = RW::valid(ln, q) ? fabs(-jac_at(q, r, j) + (d ? dr : 0.0)) + (d ? di : 0.0) : 0.0;
      int e = kZero;
      if (m > 0.0) frexp(m, &e);
      return e;
    };
#pragma unroll
    for (int q = 0; q < R; ++q) cx[q] = 0;
    int rx[R];
#pragma unroll 1
    for (int sweep = 0; sweep <= kEquilSweeps; ++sweep) {
      // row maxima under the current column scaling
      int m[R];
#pragma unroll
      for (int q = 0; q < R; ++q) m[q] = kZero;
      // (rolled loops: the sweeps are a small part of the work, and fully
      // unrolled they added code that cost the 54-state kernel 75 %)
#pragma unroll 4
      for (int j = 0; j < N; ++j) {
        const int cj = col_exp(cx, j);
#pragma unroll
        for (int q = 0; q < R; ++q) m[q] = max(m[q], eps(q, j) - cj);
      }
      const bool last = sweep == kEquilSweeps;
#pragma unroll
      for (int q = 0; q < R; ++q) rx[q] = last ? m[q] : m[q] / 2;
      if (last) break;
      // column maxima under that row scaling (a group maximum per column);
      // the lane holding row j keeps column j's exponent
      auto column = [&](int j, int cj) {
        int v = kZero;
#pragma unroll
        for (int q = 0; q < R; ++q) v = max(v, eps(q, j) - rx[q] - cj);
        float vf = (float)v;  // exact: |v| < 2^24
        int key = 0;
        group_argmax<G>(vf, key);
        const int add = (int)vf / 2;
#pragma unroll
        for (int q = 0; q < R; ++q) cx[q] = (RW::row(ln, q) == j) ? cx[q] + add : cx[q];
      };
#pragma unroll 2
      for (int j = 0; j < N; ++j) column(j, col_exp(cx, j));
    }
#pragma unroll
    for (int q = 0; q < R; ++q) ex[q] = rx[q];
  }

  // RK_Decomp, radau2a.c:256-278: E1 = gamma/H - J, E2 = (alpha + i beta)/H - J,
  // then the real and (if E1 is regular) the complex LU.  Returns info.  The
  // complex factorization also runs when E1 is singular (its info is then
  // ignored, as the reference skips it): that keeps E2 defined on every path.
  __device__ __forceinline__ int decomp(Ctx& ctx) {
    const int ln = Grp<G>::lane();
    const double iH = 1.0 / H;
    const double g1 = quot(rkGamma, H, iH), g2r = quot(rkAlpha, H, iH), g2i = quot(rkBeta, H, iH);
    int info = 0, info2 = 0;
    if constexpr (Mech::kJacInLds) group_lds_sync();
    auto jac_at = [&](int q, int r, int j) -> double {
      if constexpr (Mech::kJacInLds) return jac_entry(ctx, ln, q, j);
      else return A[q][j];
    };
    if constexpr (kMixed && kMemLU) {
      equilibrate(jac_at, g1, 0.0, ex1, cx1);
      equilibrate(jac_at, g2r, g2i, ex2, cx2);
    } else if constexpr (kMixed) {
      int e1[R], e2[R];
      row_exponents(jac_at, g1, 0.0, e1);
      row_exponents(jac_at, g2r, g2i, e2);
#pragma unroll
      for (int q = 0; q < R; ++q) ex1[q] = (int)(((unsigned)e1[q] & 0xffffu) | ((unsigned)e2[q] << 16));
    }
    // entry (r, j) of a matrix scaled by 2^-(e + c_j): c_j is held by the
    // lane that holds row j
    auto scaled = [&](double v, int e, int cj) -> MT { return kMixed ? (MT)ldexp(v, -(e + cj)) : (MT)v; };
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = RW::row(ln, q);
      const int e1 = kMixed ? row_exp1(q) : 0, e2 = kMixed ? row_exp2(q) : 0;
      if constexpr (kMemLU) {
        MT* w1 = wE1() + r;
        MT* w2r = wE2r() + r;
        MT* w2i = wE2i() + r;
#pragma unroll 16
        for (int j = 0; j < N; ++j) {
          // the column exponents are read across lanes (readlane), so with
          // every lane active: inside a branch on the row's validity the
          // lanes holding rows beyond N would not have computed them
          const int c1 = kMixed ? col_exp(cx1, j) : 0, c2 = kMixed ? col_exp(cx2, j) : 0;
          const bool d = (j == r);
          const double aj = jac_at(q, r, j);
          if (RW::valid(ln, q)) {
            w1[(size_t)j * MLU::LD] = scaled(-aj + (d ? g1 : 0.0), e1, c1);
            w2r[(size_t)j * MLU::LD] = scaled(-aj + (d ? g2r : 0.0), e2, c2);
            w2i[(size_t)j * MLU::LD] = scaled(d ? g2i : 0.0, e2, c2);
          }
        }
      } else {
        // (mixed: J' is column-scaled already; the diagonal takes its own
        // column's scale)
        const double d1 = kMixed ? ldexp(g1, -cx1[q]) : g1;
        const double d2r = kMixed ? ldexp(g2r, -cx1[q]) : g2r, d2i = kMixed ? ldexp(g2i, -cx1[q]) : g2i;
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const bool d = (j == r);
          const double aj = jac_at(q, r, j);
          E1[q][j] = scaled(-aj + (d ? d1 : 0.0), e1, 0);
          E2r[q][j] = scaled(-aj + (d ? d2r : 0.0), e2, 0);
          E2i[q][j] = scaled(d ? d2i : 0.0, e2, 0);
        }
      }
    }
    if constexpr (kMemLU) {
      wave_vmem_sync();  // every lane's rows before the panels read them
      MLU::factor_real(wE1(), wperm1(), MLU::tmp(ws), info);
      MLU::factor_cplx(wE2r(), wE2i(), wperm2(), MLU::tmp(ws), info2);
    } else if constexpr (kRow16) {
      row16_lu_real<N, MT>(E1[0], src1, rd1[0], info);
      row16_lu_cplx<N, MT>(E2r[0], E2i[0], src2, rd2r[0], rd2i[0], info2);
    } else if constexpr (G == 64 && R == 1) {
      wave_lu<N, MT>(E1, pos1, perm1, rd1, info, E2r, E2i, pos2, perm2, rd2r, rd2i, info2);
    } else {
      lu_real<N, G, R, MT>(E1, pos1, perm1, rd1, info);
      lu_cplx<N, G, R, MT>(E2r, E2i, pos2, perm2, rd2r, rd2i, info2);
    }
    return info != 0 ? info : info2;
  }

  // RK_ErrorNorm, radau2a.c:446-453: max(sqrt(sum (sc d)^2 / N), 1e-10).
  // A NaN norm is returned as +inf: fmax would turn it into 1e-10 and let a
  // non-finite Newton increment or error estimate pass as converged/accepted
  // (the reference's fmax does exactly that); +inf makes it a divergence and
  // a rejection instead.  Finite norms are unchanged.
  __device__ __forceinline__ double err_norm(const double (&d)[R]) const {
    const int ln = Grp<G>::lane();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (RW::valid(ln, q)) s += sc[q] * sc[q] * d[q] * d[q];
    s = Grp<G>::sum(s);
    const double e = sqrt(quot(s, (double)N, 1.0 / (double)N));
    return e == e ? fmax(e, 1e-10) : __builtin_inf();
  }
  // The root mean square of the three stages' norms (the Newton increment,
  // radau2a.c:640-645): from the sums of squares under the norms' floor, with one
  // root and one division instead of four each.
  __device__ __forceinline__ double err_norm3(const double (&d1)[R], const double (&d2)[R], const double (&d3)[R]) const {
    const int ln = Grp<G>::lane();
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (RW::valid(ln, q)) {
        const double w = sc[q] * sc[q];
        s1 += w * d1[q] * d1[q];
        s2 += w * d2[q] * d2[q];
        s3 += w * d3[q] * d3[q];
      }
    Grp<G>::sum3(s1, s2, s3);
    constexpr double floor_ = 1e-20 * N;
    const double e = sqrt(quot(fmax(s1, floor_) + fmax(s2, floor_) + fmax(s3, floor_), 3.0 * N, 1.0 / (3.0 * N)));
    return s1 + s2 + s3 == s1 + s2 + s3 ? e : __builtin_inf();  // (fmax drops a NaN)
  }

  // integrate() prologue, radau2a.c:521-564: a fresh start for every interval.
  __device__ __forceinline__ void begin(const SolverParams& P, double t_start, double t_stop) {
    Hold = 0.0; Hacc = 0.0; ErrOld = 0.0;
    H = P.const_time_step ? (t_stop - t_start) : fmin(5e-7, t_stop - t_start);
    t = t_start;
    t_end = t_stop;
    Reject = false; FirstStep = true; SkipJac = false; SkipLU = false;
    UseStart = false;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      sc[q] = 1.0 / (P.atol + fabs(y[q]) * P.rtol);  // scale_init, :88-94
      y0[q] = y[q];
      F0[q] = 0.0; Z1[q] = 0.0; Z2[q] = 0.0; Z3[q] = 0.0;
      CONT0[q] = 0.0; CONT1[q] = 0.0; CONT2[q] = 0.0;
    }
    Nconsecutive = 0;
    Nsteps = 0;

    NewtonRate = 2.3784142300054421;  // pow(2.0, 1.25)
  }

  __device__ __forceinline__ bool finished() const { return !(t + kRoundoff < t_end); }

  // Training sample of the learned start: features (of y at the step start,
  // log h, log pr) and the converged stages of an accepted first step.
  __device__ __forceinline__ void log_first_step(const StartLog& L, double pr) const {
    const int ln = Grp<G>::lane();
    int slot = 0;
    if (ln == 0) slot = atomicAdd(L.count, 1);
    slot = Grp<G>::bcast_i(slot, 0);
    if (slot >= L.cap) return;
    float* x = L.x + (size_t)slot * (N + 2);
    float* z = L.z + (size_t)slot * 3 * N;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (RW::valid(ln, q)) {
        const int r = RW::row(ln, q);
        x[r] = mlp_feature(r, y[q]);
        z[r] = (float)Z1[q];
        z[N + r] = (float)Z2[q];
        z[2 * N + r] = (float)Z3[q];
      }
    }
    if (ln == 0) {
      x[N] = (float)log(H);
      x[N + 1] = (float)log(pr);
    }
  }

  // One pass of the step loop, radau2a.c:566-734.  Returns RADAU_CONTINUE,
  // EC_success once t has reached t_end, or an error code.
  __device__ __forceinline__ int attempt(Ctx& ctx, const SolverParams& P, double pr, uint32_t (&cnt)[NCNT]) {
    const int ln = Grp<G>::lane();
    const double atol = P.atol, rtol = P.rtol;
    if (!Reject) {
      Mech::template dydt<G, R>(ctx, t, pr, y, F0);
      cnt[CNT_F]++;
    }
    if (!SkipLU) {
      if (!SkipJac) {
        if constexpr (Mech::kJacInLds) {
          if constexpr (JacBatched<Mech>::value)
            Mech::template jacob<G, R, kMixed && G == 64 ? Mech::kJacBatchFP32 : Mech::kJacBatchFP64>(ctx, t, pr, y);
          else
            Mech::template jacob<G, R>(ctx, t, pr, y);
        } else {
          Mech::template jacob<G, R>(ctx, t, pr, y, A);
        }
        cnt[CNT_JAC]++;
        if constexpr (kMixed && !kMemLU) park_column_scaling(ctx);
      }
      const int info = decomp(ctx);
      cnt[CNT_LU]++;
      if (info != 0) {
        cnt[CNT_LU_FAIL]++;
        UseStart = false;
        Nconsecutive += 1;
        if (Nconsecutive >= kMaxConsecutiveErrs) return EC_consecutive_steps;
        H *= 0.5;
        Reject = true;
        SkipJac = true;
        SkipLU = false;
        return RADAU_CONTINUE;
      } else {
        Nconsecutive = 0;
      }
    }
    Nsteps += 1;
    cnt[CNT_STEP]++;
    if (Nsteps >= (kMixed && kMemLU ? kMixedMaxSteps : kMaxNoSteps)) return EC_max_steps_exceeded;
    if (0.1 * fabs(H) <= fabs(t) * kRoundoff) return EC_h_plus_t_equals_h;
    if (FirstStep) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        Z1[q] = UseStart ? zs[q * G + ln] : 0.0;
        Z2[q] = UseStart ? zs[(R + q) * G + ln] : 0.0;
        Z3[q] = UseStart ? zs[(2 * R + q) * G + ln] : 0.0;
      }
    } else {
      // RK_Interpolate, :302-314 (third stage keeps the reference's x2 factor)
      const double rr = H / Hold;
      const double x1 = 1.0 + rkC0 * rr, x2 = 1.0 + rkC1 * rr, x3 = 1.0 + rkC2 * rr;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        Z1[q] = CONT0[q] + x1 * (CONT1[q] + x1 * CONT2[q]);
        Z2[q] = CONT0[q] + x2 * (CONT1[q] + x2 * CONT2[q]);
        Z3[q] = CONT0[q] + x2 * (CONT1[q] + x3 * CONT2[q]);
      }
    }
    const double iH = 1.0 / H;
    bool NewtonDone = false;
    double NewtonIncrementOld = 0.0;
    double Fac = 0.5;
    int NewtonIter = 0;
    double Theta = 0.0;
    NewtonRate = pow_0p8(fmax(NewtonRate, kRoundoff));

#pragma unroll 1
    for (; NewtonIter < kNewtonMaxit; NewtonIter++) {
      double DZ1[R], DZ2[R], DZ3[R];
      // RK_PrepareRHS, :353-383: R_k = Z_k - H sum_j A_kj f(t + c_j H, y + Z_j),
      // one callback site for the three stage evaluations
#pragma unroll
      for (int q = 0; q < R; ++q) { DZ1[q] = Z1[q]; DZ2[q] = Z2[q]; DZ3[q] = Z3[q]; }
#pragma unroll 1
      for (int js = 0; js < 3; ++js) {
        double Tm[R], F[R];
#pragma unroll
        for (int q = 0; q < R; ++q) Tm[q] = y[q] + (js == 0 ? Z1[q] : (js == 1 ? Z2[q] : Z3[q]));
        const double cj = js == 0 ? rkC0 : (js == 1 ? rkC1 : rkC2);
        Mech::template dydt<G, R>(ctx, t + cj * H, pr, Tm, F);
        const double a1 = -H * (js == 0 ? rkA00 : (js == 1 ? rkA01 : rkA02));
        const double a2 = -H * (js == 0 ? rkA10 : (js == 1 ? rkA11 : rkA12));
        const double a3 = -H * (js == 0 ? rkA20 : (js == 1 ? rkA21 : rkA22));
#pragma unroll
        for (int q = 0; q < R; ++q) { DZ1[q] += a1 * F[q]; DZ2[q] += a2 * F[q]; DZ3[q] += a3 * F[q]; }
      }
      cnt[CNT_F] += 3;
      // RK_Solve, :388-441
      {
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const double x1 = quot(DZ1[q], H, iH), x2 = quot(DZ2[q], H, iH), x3 = quot(DZ3[q], H, iH);
          DZ1[q] = rkTiAi00 * x1 + rkTiAi01 * x2 + rkTiAi02 * x3;
          DZ2[q] = rkTiAi10 * x1 + rkTiAi11 * x2 + rkTiAi12 * x3;
          DZ3[q] = rkTiAi20 * x1 + rkTiAi21 * x2 + rkTiAi22 * x3;
        }
        // (interleaving the real and complex substitutions was measured
        // slower in this kernel: the larger live set spills)
        solve1(DZ1);
        solve2(DZ2, DZ3);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const double x1 = DZ1[q], x2 = DZ2[q], x3 = DZ3[q];
          DZ1[q] = rkT00 * x1 + rkT01 * x2 + rkT02 * x3;
          DZ2[q] = rkT10 * x1 + rkT11 * x2 + rkT12 * x3;
          DZ3[q] = rkT20 * x1 + rkT21 * x2 + rkT22 * x3;
        }
        cnt[CNT_NEWTON]++;
      }
      const double NewtonIncrement = err_norm3(DZ1, DZ2, DZ3);
      if (FirstStep && UseStart && NewtonIter == 0) {
        // A predicted start is kept only if its first Newton correction is
        // smaller than the corrected stages, i.e. than the zero start's
        // distance from the same point; otherwise Newton restarts from zero.
        double W1[R], W2[R], W3[R];
#pragma unroll
        for (int q = 0; q < R; ++q) { W1[q] = Z1[q] - DZ1[q]; W2[q] = Z2[q] - DZ2[q]; W3[q] = Z3[q] - DZ3[q]; }
        if (!(NewtonIncrement < err_norm3(W1, W2, W3))) {
          UseStart = false;
          StartFailed = true;
#pragma unroll
          for (int q = 0; q < R; ++q) { Z1[q] = 0.0; Z2[q] = 0.0; Z3[q] = 0.0; }
          NewtonIter = -1;  // the loop's increment makes the restart iteration 0
          continue;
        }
      }
      Theta = kThetaMin;
      if (NewtonIter > 0) {
        Theta = NewtonIncrement / NewtonIncrementOld;
        if (Theta < 0.99) {
          NewtonRate = Theta / (1.0 - Theta);
        } else {
          break;
        }
        const double NewtonPredictedErr =
            (NewtonIncrement * pow_int(Theta, kNewtonMaxit - NewtonIter - 1)) / (1.0 - Theta);
        if (NewtonPredictedErr >= kNewtonTol) {
          const double Qnewton = fmin(10.0, NewtonPredictedErr / kNewtonTol);
          Fac = 0.8 * step_pow(Qnewton, -1.0 / ((double)(kNewtonMaxit - NewtonIter)));
          break;
        }
      }
      NewtonIncrementOld = fmax(NewtonIncrement, kRoundoff);
#pragma unroll
      for (int q = 0; q < R; ++q) { Z1[q] -= DZ1[q]; Z2[q] -= DZ2[q]; Z3[q] -= DZ3[q]; }
      // With FP32 factors the iteration is only linearly convergent, at a rate
      // that depends on the factors' accuracy: convergence is declared only
      // on a contraction rate measured in this step (from the second
      // iteration on), never on the rate carried over from the previous step.
      NewtonDone = (!kMixed || NewtonIter > 0) && (NewtonRate * NewtonIncrement <= kNewtonTol);
      if (NewtonDone) break;
      if (NewtonIter == kNewtonMaxit - 1) {
        if (FirstStep && UseStart) break;
        return EC_newton_max_iterations_exceeded;
      }
    }
    if (!NewtonDone && FirstStep && UseStart) {
      // A predicted start that does not converge falls back to the zero
      // start at the same H; the factorizations belong to this H and are kept.
      cnt[CNT_NEWTON_FAIL]++;
      UseStart = false;
      StartFailed = true;
      SkipJac = true;
      SkipLU = true;
      return RADAU_CONTINUE;
    }
    // Fallback by iteration count: a predicted start that needed three or
    // more Newton iterations did no better than the zero start typically does
    // on this step (two or more, three at the median), so the condition
    // stops predicting for the rest of the call, as after a discarded start.
    if (FirstStep && UseStart && NewtonIter >= 2) StartFailed = true;
    if (P.const_time_step) {  // :725-733
      t += H;
#pragma unroll
      for (int q = 0; q < R; ++q) y[q] += Z3[q];
      cnt[CNT_ACCEPT]++;
      return finished() ? EC_success : RADAU_CONTINUE;
    }
    if (!NewtonDone) {
      cnt[CNT_NEWTON_FAIL]++;
      UseStart = false;
      H = Fac * H;
      Reject = true;
      SkipJac = true;
      SkipLU = false;
      return RADAU_CONTINUE;
    }
    // RK_ErrorEstimate, :458-508: solve E1 x = e0 F0 + F2; on a first or
    // rejected step with Err >= 1, solve again with f(t, y + x) + F2.
    double Err;
    {
      const double HrkE1 = quot(rkE1, H, iH), HrkE2 = quot(rkE2, H, iH), HrkE3 = quot(rkE3, H, iH);
      double F2[R], Tm[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        F2[q] = HrkE1 * Z1[q] + HrkE2 * Z2[q] + HrkE3 * Z3[q];
        Tm[q] = rkE0 * F0[q] + F2[q];
      }
#pragma unroll 1
      for (int pass = 0;; ++pass) {
        solve1_es(ctx, Tm);
        cnt[CNT_ES]++;
        Err = err_norm(Tm);
        if (pass == 1 || !(Err >= 1.0 && (FirstStep || Reject))) break;
        double F1[R];
#pragma unroll
        for (int q = 0; q < R; ++q) Tm[q] += y[q];
        Mech::template dydt<G, R>(ctx, t, pr, Tm, F1);
        cnt[CNT_F]++;
#pragma unroll
        for (int q = 0; q < R; ++q) Tm[q] = F1[q] + F2[q];
      }
    }
    Fac = inv_root4(Err) * (1.0 + 2 * kNewtonMaxit) / (NewtonIter + 1.0 + 2 * kNewtonMaxit);
    Fac = fmin(kFacMax, fmax(kFacMin, Fac));
    double Hnew = Fac * H;
    if (Err < 1.0) {
      cnt[CNT_ACCEPT]++;
      if (FirstStep && P.log.cap > 0) log_first_step(P.log, pr);
      if (!FirstStep) {  // Gustafsson, :676-685
        double FacGus = kFacSafe * (H / Hacc) * inv_root4(Err * Err / ErrOld);
        FacGus = fmin(kFacMax, fmax(kFacMin, FacGus));
        Fac = fmin(Fac, FacGus);
        Hnew = Fac * H;
      }
      Hacc = H;
      ErrOld = fmax(1e-2, Err);
      FirstStep = false;
      Hold = H;
      t += H;
#pragma unroll
      for (int q = 0; q < R; ++q) y[q] += Z3[q];
      // RK_Make_Interpolate, :283-297
      {
        constexpr double den = (rkC2 - rkC1) * (rkC1 - rkC0) * (rkC0 - rkC2), iden = 1.0 / den;
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const double z1 = Z1[q], z2 = Z2[q], z3 = Z3[q];
          CONT0[q] = quot(-rkC2 * rkC2 * rkC1 * z1 + z3 * rkC1 * rkC0 * rkC0 + rkC1 * rkC1 * rkC2 * z1 -
                              rkC1 * rkC1 * rkC0 * z3 + rkC2 * rkC2 * rkC0 * z2 - z2 * rkC2 * rkC0 * rkC0,
                          den, iden) - z3;
          CONT1[q] = -quot(rkC0 * rkC0 * (z3 - z2) + rkC1 * rkC1 * (z1 - z3) + rkC2 * rkC2 * (z2 - z1), den, iden);
          CONT2[q] = quot(rkC0 * (z3 - z2) + rkC1 * (z1 - z3) + rkC2 * (z2 - z1), den, iden);
        }
      }
#pragma unroll
      for (int q = 0; q < R; ++q) {  // scale(), :74-81
        sc[q] = 1.0 / (atol + fmax(fabs(y[q]), fabs(y0[q])) * rtol);
        y0[q] = y[q];
      }
      Hnew = fmin(fmax(Hnew, 0.0), t_end - t);  // Hmin = 0
      if (Reject) Hnew = fmin(Hnew, H);
      Reject = false;
      if (t + Hnew / kQmin - t_end >= 0.0) {
        H = t_end - t;
      } else {
        const double Hratio = Hnew / H;
        SkipLU = (Theta <= kThetaMin) && (Hratio >= kQmin) && (Hratio <= kQmax);
        if (!SkipLU) H = Hnew;
      }
      SkipJac = NewtonIter == 1 || NewtonRate <= kThetaMin;
      return finished() ? EC_success : RADAU_CONTINUE;
    } else {
      cnt[CNT_REJECT]++;
      UseStart = false;
      if (FirstStep || Reject) {
        H = kFacRej * H;
      } else {
        H = Hnew;
      }
      Reject = true;
      SkipJac = true;
      SkipLU = false;
      return RADAU_CONTINUE;
    }
  }
};

}  // namespace acc
