// Iteration-matrix factorizations of large systems (N > 64): one wavefront
// per condition, R rows per lane (row r = lane + 64 q), the real and complex
// matrices in a per-wave global workspace that stays in L2 / the MALL,
// column-major E[j * LD + i] with LD = 64 R.
//
// dgetrf / zgetrf semantics (the reference's RK_Decomp, radau2a.c:256-278,
// through LAPACK): partial pivoting on the first maximum of |a| (real) or
// |Re| + |Im| (complex), blocked right-looking with implicit interchanges --
// rows stay where they are, each records the LAPACK position it would hold --
// until one gather at the end puts them in order:
//   1. the panel of 16 columns is factorized in registers (each lane holds its
//      rows' 16 panel entries; one-word pivot search, the pivot row broadcast
//      through SGPRs);
//   2. the pivot rows' trailing part is solved against the panel's unit-lower
//      block (dtrsm), lanes over columns;
//   3. the trailing matrix takes the rank-16 update A22 -= L21 U12 on MFMA
//      (v_mfma_{f32,f64}_16x16x4: four K = 4 steps per 16 x 16 tile; complex:
//      four real products per step) over all row tiles, the rows already
//      eliminated with zero multipliers: L21 (so masked) and U12 are taken from
//      copies laid out for the operands, all of a column tile's loads are in
//      flight together and L21 stays in registers for the whole panel.
// Within a wave, global stores made by one lane are read by other lanes only
// after s_waitcnt vmcnt(0): the wave's vector memory traffic goes through its
// CU's write-through L1, so that wait makes them visible on the same CU.
// The solves (dgetrs / zgetrs, radau2a.c:404,417) gather the right-hand side
// and substitute column by column, skipping zero entries as reference BLAS
// does, with the next block of columns loaded while one is used.
//
// Bound by latency: a single wave, workspace in L2.  With explicit interchanges
// (a panel's 16 composed by wave-uniform index work and applied column by
// column, 64 cache lines an access) and two row tiles in flight, an FP64 pair
// took 4.8M cycles and the two solves 0.23M and 0.27M; now 1.7M, 0.07M and 0.12M
// (24 112-state conditions beside 2049 54-state and 8190 14-state ones, one step in
// FP64: 361.6 -> 131.9 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace acc {

__device__ __forceinline__ void wave_vmem_sync() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// D = A B + D on one 16 x 16 tile (A 16 x 4: lane l holds A[l % 16][l / 16];
// B 4 x 16: lane l holds B[l / 16][l % 16]; D: lane l holds column l % 16 of
// four rows, d_row(l / 16, i) for i = 0..3: rows 4 (l / 16) + i for
// v_mfma_f32_16x16x4f32 and rows l / 16 + 4 i for v_mfma_f64_16x16x4f64, as
// measured on gfx950 (a = lane, b = 1 gives row sums; a = 1, b = lane column
// sums).
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
typedef double mfma_d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mfma_f4 mfma16x16x4(float a, float b, mfma_f4 d) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0);
}
__device__ __forceinline__ mfma_d4 mfma16x16x4(double a, double b, mfma_d4 d) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, d, 0, 0, 0);
}
template <class T>
using mfma_vec = typename std::conditional<std::is_same<T, float>::value, mfma_f4, mfma_d4>::type;
template <class T>
__device__ __forceinline__ constexpr int d_row(int lq, int i) {
  return std::is_same<T, float>::value ? 4 * lq + i : lq + 4 * i;
}

template <int N, int R, class T>
struct MemLU {
  static constexpr int LD = 64 * R;
  static constexpr int NT = N / 16;
  static constexpr size_t kMat = (size_t)LD * N;  // elements of one matrix
  static_assert(N % 16 == 0 && N > 64 && N <= LD, "memory LU: N a multiple of 16 in (64, 64 R]");
  // workspace: E1, E2r, E2i (T, kMat each), then perm1[N], perm2[N] (int: the
  // original row in each position), then a factorization's temporaries: L21
  // (16 columns of LD) and U12 (16 entries per column), real and imaginary
  static constexpr size_t kTmpL = (size_t)16 * LD, kTmpU = (size_t)16 * N;
  __host__ __device__ static constexpr size_t bytes() {
    return (3 * kMat + 2 * (kTmpL + kTmpU)) * sizeof(T) + 2 * (size_t)N * sizeof(int);
  }
  __device__ __forceinline__ static int* perm1(T* ws) { return reinterpret_cast<int*>(ws + 3 * kMat); }
  __device__ __forceinline__ static int* perm2(T* ws) { return perm1(ws) + N; }
  __device__ __forceinline__ static T* tmp(T* ws) { return reinterpret_cast<T*>(perm1(ws) + 2 * N); }

  // (pinned: with a lane index known to be constant the compiler computes every
  // address of every phase once per kernel and keeps them in scratch)
  __device__ __forceinline__ static int lane() {
    int l = (int)__lane_id();
    pin(l);
    return l;
  }
  // uniform broadcast of row r's value v (r runtime-uniform)
  __device__ __forceinline__ static T row_value(const T (&v)[R], int r) {
    return Grp<64>::bcast(sel<R>(v, r >> 6), r & 63);
  }

  // Pivot of step c among the rows with position >= c: the row, wave-uniform.
  // The leading 32 bits of the magnitudes decide (see wave_pivot2); if no
  // candidate compares (a NaN column) the row at position c stays, as idamax
  // returns its first index when nothing compares greater.
  __device__ __forceinline__ static int pivot(const T (&v)[R], const int (&pos)[R], int c) {
    unsigned key[R], m = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      key[q] = pos[q] >= c && v[q] == v[q] ? mag_hi(v[q]) + 1u : 0u;
      m = max_u(m, key[q]);
    }
    m = dpp_max_u<kDppXor1>(m);
    m = dpp_max_u<kDppXor2>(m);
    m = dpp_max_u<kDppHalfMirror>(m);
    m = dpp_max_u<kDppMirror>(m);
    int x = (int)m, y = (int)m;
    swap_row_pairs(x, y);
    x = y = (int)max_u((unsigned)x, (unsigned)y);
    swap_halves(x, y);
    m = (unsigned)__builtin_amdgcn_readfirstlane((int)max_u((unsigned)x, (unsigned)y));
    unsigned long long cand[R];
    int n = 0, row = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      cand[q] = __builtin_amdgcn_ballot_w64(m != 0 ? key[q] == m : pos[q] == c);
      n += __builtin_popcountll(cand[q]);
      row = cand[q] ? 64 * q + (int)__builtin_ctzll(cand[q]) : row;
    }
    if (__builtin_expect(n > 1, 0)) {
      row = -1;
      T bv = T(0);
      int best = 0;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        unsigned long long w = cand[q];
        while (w) {
          const int l = (int)__builtin_ctzll(w);
          w &= w - 1;
          const T vl = Grp<64>::bcast(v[q], l);
          const int pl = __builtin_amdgcn_readlane(pos[q], l);
          if (row < 0 || vl > bv || (vl == bv && pl < best)) {
            bv = vl;
            best = pl;
            row = 64 * q + l;
          }
        }
      }
    }
    return __builtin_amdgcn_readfirstlane(row);
  }
  __device__ __forceinline__ static int row_value(const int (&v)[R], int r) {
    return Grp<64>::bcast_i(sel<R>(v, r >> 6), r & 63);
  }
  __device__ __forceinline__ static void init_pos(int (&pos)[R]) {
#pragma unroll
    for (int q = 0; q < R; ++q) pos[q] = (int)__lane_id() + 64 * q < N ? (int)__lane_id() + 64 * q : -1;
  }
  // position bookkeeping of one interchange: row p to position c
  __device__ __forceinline__ static void take(int (&pos)[R], int p, int c) {
    const int ppos = row_value(pos, p);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      pos[q] = (int)__lane_id() + 64 * q == p ? c : (pos[q] == c ? ppos : pos[q]);
      pin(pos[q]);
    }
  }

  // ---- real ------------------------------------------------------------------
  __device__ __forceinline__ static void panel_real(T* E, T* L, int k, T (&pv)[R][16], int (&pos)[R], int (&piv)[16],
                                                    int& info) {
    const int ln = lane();
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int c = 0; c < 16; ++c) pv[q][c] = E[(size_t)(k + c) * LD + ln + 64 * q];  // rows up to LD are in the workspace
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const int c = k + kk;
      T mag[R], col[R];
#pragma unroll
      for (int q = 0; q < R; ++q) mag[q] = fabs(pv[q][kk]);
      const int p = pivot(mag, pos, c);
      piv[kk] = p;
      take(pos, p, c);
#pragma unroll
      for (int q = 0; q < R; ++q) col[q] = pv[q][kk];
      const T pval = row_value(col, p);
      const bool nz = !is_zero(pval);
      info = !nz && info == 0 ? c + 1 : info;
      const T rp = recip(pval);
      const bool tiny = std::is_same<T, double>::value && fabs(pval) < min_normal<T>();
      T l[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        T v = pv[q][kk] * rp;
        if (__builtin_expect(tiny, 0)) v = pv[q][kk] / pval;
        // (with a zero pivot the column's active part is zero: nothing to add)
        const bool act = nz && pos[q] > c;
        pv[q][kk] = act ? v : pv[q][kk];
        l[q] = act ? -v : T(-0.0);
        pin(pv[q][kk]);
        pin(l[q]);
      }
#pragma unroll
      for (int c2 = kk + 1; c2 < 16; ++c2) {
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] = pv[q][c2];
        const T u = row_value(col, p);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          pv[q][c2] = fma(l[q], u, pv[q][c2]);
          pin(pv[q][c2]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + 64 * q;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        E[(size_t)(k + c) * LD + r] = pv[q][c];
        L[(size_t)c * LD + r] = pos[q] >= k + 16 ? -pv[q][c] : T(0);
      }
    }
  }

  // U12 = L11^-1 A12 on the 16 pivot rows, columns k+16 .. N-1 (lanes over
  // columns), into the matrix and, 16 entries per column, into U
  __device__ __forceinline__ static void trsm_real(T* E, T* U, int k, const T (&pv)[R][16], const int (&piv)[16]) {
    const int ln = lane();
    constexpr int M = (N + 63) / 64;
    T u[M][16];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int j = min(k + 16 + ln + 64 * m, N - 1);
#pragma unroll
      for (int i = 0; i < 16; ++i) u[m][i] = E[(size_t)j * LD + piv[i]];
    }
#pragma unroll
    for (int i = 1; i < 16; ++i) {
#pragma unroll
      for (int mm = 0; mm < i; ++mm) {
        T col[R];
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] = pv[q][mm];
        const T lim = row_value(col, piv[i]);  // L(k+i, k+mm)
#pragma unroll
        for (int m = 0; m < M; ++m) u[m][i] = fma(-lim, u[m][mm], u[m][i]);
      }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int j = k + 16 + ln + 64 * m;
      if (j < N) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          U[(size_t)j * 16 + i] = u[m][i];
          if (i > 0) E[(size_t)j * LD + piv[i]] = u[m][i];
        }
      }
    }
  }

  // A22 -= L21 U12 (columns k+16 .. N-1, all rows) on MFMA
  __device__ __forceinline__ static void update_real(T* E, const T* L, const T* U, int k) {
    const int ln = lane(), lr = ln & 15, lq = ln >> 4;
    T a[NT][4];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt)
#pragma unroll
      for (int t = 0; t < 4; ++t) a[rt][t] = L[(size_t)(4 * t + lq) * LD + rt * 16 + lr];
#pragma unroll 1
    for (int cb = k / 16 + 1; cb < NT; ++cb) {
      T* ccol = E + (size_t)(cb * 16 + lr) * LD;
      T b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = U[(size_t)(cb * 16 + lr) * 16 + 4 * t + lq];
      mfma_vec<T> acc[NT];
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][i] = ccol[rt * 16 + d_row<T>(lq, i)];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) acc[rt] = mfma16x16x4(a[rt][t], b[t], acc[rt]);
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) ccol[rt * 16 + d_row<T>(lq, i)] = acc[rt][i];
    }
  }

  // rows into their positions (perm: the original row of every position)
  __device__ __forceinline__ static void order_rows(T* E, const int* perm) {
    const int ln = lane();
    int src[R];
#pragma unroll
    for (int q = 0; q < R; ++q) src[q] = perm[min(ln + 64 * q, N - 1)];
#pragma unroll 1
    for (int j0 = 0; j0 < N; j0 += 16) {
      T v[R][16];
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int c = 0; c < 16; ++c) v[q][c] = E[(size_t)(j0 + c) * LD + src[q]];
      wave_vmem_sync();  // every lane has read before any writes
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int c = 0; c < 16; ++c) E[(size_t)(j0 + c) * LD + ln + 64 * q] = v[q][c];
    }
  }

  __device__ __forceinline__ static void store_piv(int* perm, int k, const int (&piv)[16]) {
    if (lane() == 0) {
#pragma unroll
      for (int kk = 0; kk < 16; ++kk) perm[k + kk] = piv[kk];
    }
  }

  __device__ static void factor_real(T* E, int* perm, T* tmp, int& info) {
    T *L = tmp, *U = tmp + kTmpL;
    int pos[R];
    init_pos(pos);
    info = 0;
#pragma unroll 1
    for (int k = 0; k < N; k += 16) {
      T pv[R][16];
      int piv[16];
      panel_real(E, L, k, pv, pos, piv, info);
      store_piv(perm, k, piv);
      if (k + 16 < N) {
        wave_vmem_sync();
        trsm_real(E, U, k, pv, piv);
        wave_vmem_sync();
        update_real(E, L, U, k);
      }
      wave_vmem_sync();
    }
    order_rows(E, perm);
    wave_vmem_sync();
  }

  // ---- complex ---------------------------------------------------------------
  __device__ __forceinline__ static void panel_cplx(T* Er, T* Ei, T* Lr, T* Li, int k, T (&pr)[R][16], T (&pi)[R][16],
                                                    int (&pos)[R], int (&piv)[16], int& info) {
    const int ln = lane();
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        pr[q][c] = Er[(size_t)(k + c) * LD + ln + 64 * q];
        pi[q][c] = Ei[(size_t)(k + c) * LD + ln + 64 * q];
      }
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const int c = k + kk;
      T mag[R], cr[R], ci[R];
#pragma unroll
      for (int q = 0; q < R; ++q) mag[q] = fabs(pr[q][kk]) + fabs(pi[q][kk]);
      const int p = pivot(mag, pos, c);
      piv[kk] = p;
      take(pos, p, c);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        cr[q] = pr[q][kk];
        ci[q] = pi[q][kk];
      }
      const T vr = row_value(cr, p), vi = row_value(ci, p);
      const bool nz = !(is_zero(vr) && is_zero(vi));
      info = !nz && info == 0 ? c + 1 : info;
      T rr, ri;
      crecip(vr, vi, rr, ri);
      T lr[R], li[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const T xr = pr[q][kk], xi = pi[q][kk];
        const T sr = xr * rr - xi * ri, si = xr * ri + xi * rr;
        const bool act = nz && pos[q] > c;
        pr[q][kk] = act ? sr : xr;
        pi[q][kk] = act ? si : xi;
        lr[q] = act ? sr : T(0);
        li[q] = act ? si : T(0);
        pin(pr[q][kk]);
        pin(pi[q][kk]);
        pin(lr[q]);
        pin(li[q]);
      }
#pragma unroll
      for (int c2 = kk + 1; c2 < 16; ++c2) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
          cr[q] = pr[q][c2];
          ci[q] = pi[q][c2];
        }
        const T ur = row_value(cr, p), ui = row_value(ci, p);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          pr[q][c2] = fma(li[q], ui, fma(-lr[q], ur, pr[q][c2]));
          pi[q][c2] = fma(-li[q], ur, fma(-lr[q], ui, pi[q][c2]));
          pin(pr[q][c2]);
          pin(pi[q][c2]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + 64 * q;
      const bool below = pos[q] >= k + 16;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        Er[(size_t)(k + c) * LD + r] = pr[q][c];
        Ei[(size_t)(k + c) * LD + r] = pi[q][c];
        Lr[(size_t)c * LD + r] = below ? pr[q][c] : T(0);
        Li[(size_t)c * LD + r] = below ? pi[q][c] : T(0);
      }
    }
  }

  __device__ __forceinline__ static void trsm_cplx(T* Er, T* Ei, T* Ur, T* Ui, int k, const T (&pr)[R][16],
                                                   const T (&pi)[R][16], const int (&piv)[16]) {
    const int ln = lane();
    constexpr int M = (N + 63) / 64;
#pragma unroll 1
    for (int m = 0; m < M; ++m) {
      if (k + 16 + 64 * m >= N) break;
      const int j = k + 16 + ln + 64 * m, jj = min(j, N - 1);
      T ur[16], ui[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        ur[i] = Er[(size_t)jj * LD + piv[i]];
        ui[i] = Ei[(size_t)jj * LD + piv[i]];
      }
#pragma unroll
      for (int i = 1; i < 16; ++i) {
#pragma unroll
        for (int mm = 0; mm < i; ++mm) {
          T cr[R], ci[R];
#pragma unroll
          for (int q = 0; q < R; ++q) {
            cr[q] = pr[q][mm];
            ci[q] = pi[q][mm];
          }
          const T lr = row_value(cr, piv[i]), li = row_value(ci, piv[i]);
          ur[i] = fma(-lr, ur[mm], ur[i]);
          ur[i] = fma(li, ui[mm], ur[i]);
          ui[i] = fma(-lr, ui[mm], ui[i]);
          ui[i] = fma(-li, ur[mm], ui[i]);
        }
      }
      if (j < N) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          Ur[(size_t)j * 16 + i] = ur[i];
          Ui[(size_t)j * 16 + i] = ui[i];
          if (i > 0) {
            Er[(size_t)j * LD + piv[i]] = ur[i];
            Ei[(size_t)j * LD + piv[i]] = ui[i];
          }
        }
      }
    }
  }

  // (Dr + i Di) -= (Lr + i Li)(Ur + i Ui) on MFMA: Dr += (-Lr) Ur + Li Ui,
  // Di += (-Lr) Ui + (-Li) Ur
  __device__ __forceinline__ static void update_cplx(T* Er, T* Ei, const T* Lr, const T* Li, const T* Ur, const T* Ui,
                                                     int k) {
    const int ln = lane(), lr = ln & 15, lq = ln >> 4;
    T ar[NT][4], ai[NT][4];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const size_t a = (size_t)(4 * t + lq) * LD + rt * 16 + lr;
        ar[rt][t] = Lr[a];
        ai[rt][t] = Li[a];
      }
#pragma unroll 1
    for (int cb = k / 16 + 1; cb < NT; ++cb) {
      const size_t cc = (size_t)(cb * 16 + lr) * LD;
      T br[4], bi[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        br[t] = Ur[(size_t)(cb * 16 + lr) * 16 + 4 * t + lq];
        bi[t] = Ui[(size_t)(cb * 16 + lr) * 16 + 4 * t + lq];
      }
      mfma_vec<T> xr[NT], xi[NT];
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xr[rt][i] = Er[cc + rt * 16 + d_row<T>(lq, i)];
          xi[rt][i] = Ei[cc + rt * 16 + d_row<T>(lq, i)];
        }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
          xr[rt] = mfma16x16x4(-ar[rt][t], br[t], xr[rt]);
          xi[rt] = mfma16x16x4(-ar[rt][t], bi[t], xi[rt]);
        }
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
          xr[rt] = mfma16x16x4(ai[rt][t], bi[t], xr[rt]);
          xi[rt] = mfma16x16x4(-ai[rt][t], br[t], xi[rt]);
        }
      }
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          Er[cc + rt * 16 + d_row<T>(lq, i)] = xr[rt][i];
          Ei[cc + rt * 16 + d_row<T>(lq, i)] = xi[rt][i];
        }
    }
  }

  __device__ static void factor_cplx(T* Er, T* Ei, int* perm, T* tmp, int& info) {
    T *Lr = tmp, *Li = Lr + kTmpL, *Ur = Li + kTmpL, *Ui = Ur + kTmpU;
    int pos[R];
    init_pos(pos);
    info = 0;
#pragma unroll 1
    for (int k = 0; k < N; k += 16) {
      T pr[R][16], pi[R][16];
      int piv[16];
      panel_cplx(Er, Ei, Lr, Li, k, pr, pi, pos, piv, info);
      store_piv(perm, k, piv);
      if (k + 16 < N) {
        wave_vmem_sync();
        trsm_cplx(Er, Ei, Ur, Ui, k, pr, pi, piv);
        wave_vmem_sync();
        update_cplx(Er, Ei, Lr, Li, Ur, Ui, k);
      }
      wave_vmem_sync();
    }
    order_rows(Er, perm);
    order_rows(Ei, perm);
    wave_vmem_sync();
  }

  // ---- solves (nrhs = 1; b[q] = component of row lane + 64 q) ---------------
  // Every factor entry is loaded unconditionally (rows up to LD are in the
  // workspace) and the update is selected, so the next block of columns is in
  // flight while a block's columns wait for each other's broadcasts; a zero
  // right-hand-side entry skips its column, as reference BLAS does.
  __device__ __forceinline__ static void gather(const int* perm, T (&b)[R]) {
    const int ln = lane();
    T v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int src = perm[min(ln + 64 * q, N - 1)];
      v[q] = __shfl(b[0], src & 63);
#pragma unroll
      for (int p = 1; p < R; ++p) {
        const T w = __shfl(b[p], src & 63);
        v[q] = (src >> 6) == p ? w : v[q];
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) b[q] = v[q];
  }
  template <int B>
  __device__ __forceinline__ static void columns(const T* E, int k0, T (&l)[R][B]) {
    const int ln = lane();
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int i = 0; i < B; ++i) l[q][i] = E[(size_t)(k0 + i) * LD + ln + 64 * q];
  }

  __device__ static void solve_real(const T* E, const int* perm, T (&b)[R]) {
    constexpr int B = 16;
    const int ln = lane();
    T l[R][B], nx[R][B];
    columns<B>(E, 0, nx);
    gather(perm, b);
#pragma unroll 1
    for (int k0 = 0; k0 < N; k0 += B) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int i = 0; i < B; ++i) l[q][i] = nx[q][i];
      columns<B>(E, k0 + B < N ? k0 + B : N - B, nx);  // (at the end: the first block of the way back)
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int k = k0 + i;
        const T yk = row_value(b, k);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int r = ln + 64 * q;
          const T nb = fma(-l[q][i], yk, b[q]);
          b[q] = (yk != T(0) && r > k && r < N) ? nb : b[q];
        }
      }
    }
#pragma unroll 1
    for (int k0 = N - B; k0 >= 0; k0 -= B) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int i = 0; i < B; ++i) l[q][i] = nx[q][i];
      if (k0 > 0) columns<B>(E, k0 - B, nx);
#pragma unroll
      for (int i = B - 1; i >= 0; --i) {
        const int k = k0 + i;
        T col[R];
#pragma unroll
        for (int q = 0; q < R; ++q) col[q] = l[q][i];
        const T bk = row_value(b, k);
        const T xk = bk / row_value(col, k);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int r = ln + 64 * q;
          const T nb = fma(-col[q], xk, b[q]);
          b[q] = bk != T(0) ? (r < k ? nb : (r == k ? xk : b[q])) : b[q];
        }
      }
    }
  }

  __device__ static void solve_cplx(const T* Er, const T* Ei, const int* perm, T (&br)[R], T (&bi)[R]) {
    constexpr int B = 8;
    const int ln = lane();
    T lr[R][B], li[R][B], nr_[R][B], ni_[R][B];
    columns<B>(Er, 0, nr_);
    columns<B>(Ei, 0, ni_);
    gather(perm, br);
    gather(perm, bi);
#pragma unroll 1
    for (int k0 = 0; k0 < N; k0 += B) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int i = 0; i < B; ++i) {
          lr[q][i] = nr_[q][i];
          li[q][i] = ni_[q][i];
        }
      const int kn = k0 + B < N ? k0 + B : N - B;
      columns<B>(Er, kn, nr_);
      columns<B>(Ei, kn, ni_);
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int k = k0 + i;
        const T yr = row_value(br, k), yi = row_value(bi, k);
        const bool go = yr != T(0) || yi != T(0);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int r = ln + 64 * q;
          T nr = fma(-lr[q][i], yr, br[q]);
          nr = fma(li[q][i], yi, nr);
          T ni = fma(-lr[q][i], yi, bi[q]);
          ni = fma(-li[q][i], yr, ni);
          const bool act = go && r > k && r < N;
          br[q] = act ? nr : br[q];
          bi[q] = act ? ni : bi[q];
        }
      }
    }
#pragma unroll 1
    for (int k0 = N - B; k0 >= 0; k0 -= B) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int i = 0; i < B; ++i) {
          lr[q][i] = nr_[q][i];
          li[q][i] = ni_[q][i];
        }
      if (k0 > 0) {
        columns<B>(Er, k0 - B, nr_);
        columns<B>(Ei, k0 - B, ni_);
      }
#pragma unroll
      for (int i = B - 1; i >= 0; --i) {
        const int k = k0 + i;
        T cr[R], ci[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
          cr[q] = lr[q][i];
          ci[q] = li[q][i];
        }
        const T vr = row_value(br, k), vi = row_value(bi, k);
        const bool go = vr != T(0) || vi != T(0);
        // Smith's division (vr + i vi) / (dr + i di), as zgetrs divides
        T xr, xi;
        cdiv_t(vr, vi, row_value(cr, k), row_value(ci, k), xr, xi);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int r = ln + 64 * q;
          T nr = fma(-cr[q], xr, br[q]);
          nr = fma(ci[q], xi, nr);
          T ni = fma(-cr[q], xi, bi[q]);
          ni = fma(-ci[q], xr, ni);
          br[q] = go ? (r < k ? nr : (r == k ? xr : br[q])) : br[q];
          bi[q] = go ? (r < k ? ni : (r == k ? xi : bi[q])) : bi[q];
        }
      }
    }
  }

  // Smith's complex division (a + ib) / (c + id)
  __device__ __forceinline__ static void cdiv_t(T a, T b, T c, T d, T& re, T& im) {
    if (fabs(c) >= fabs(d)) {
      const T r = d / c, den = c + d * r;
      re = (a + b * r) / den;
      im = (b - a * r) / den;
    } else {
      const T r = c / d, den = c * r + d;
      re = (a * r + b) / den;
      im = (b * r - a) / den;
    }
  }
};

}  // namespace acc
