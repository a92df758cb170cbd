// Synthetic constant-pressure mass-action kinetics, dydt + analytic dense
// Jacobian, for the lane-group layout.
//
// This stands in for the pyJac-generated callbacks the reference expects in
// mechanism/ (examples/pyJac/pyJac.dox:9-33; callback contract
// examples/van_der_pol/dydt.cu:31-39, jacob.cu:31-43): state y = (T, Y_1..Y_ns),
// pr = pressure [Pa], Jacobian column-major J[i + j*N] = d f_i / d y_j, here
// delivered as the rows each lane owns.
//
// Model (all lanes of a group cooperate on one condition):
//   S = sum Y_k/W_k, Ctot = 1e-6 P/(R T) [mol/cm^3], C_k = Ctot (Y_k/W_k)/S
//   kf = exp(lnA + beta ln(T/1000) - EaR/T), ln Kc = -sum nu g/RT + dnu ln C0
//   q_j = kf prod C(reactants) - kf/Kc prod C(products)
//   dY_k/dt = W_k wdot_k S/Ctot,  dT/dt = -(sum H_k wdot_k) S/(Ctot cp)
// evaluated at T clamped to [kKinTmin, kKinTmax], S >= kKinSmin, cp >= kKinCpmin.
// Work split: species rows are owned as usual (row 0 = T, row k+1 = species
// k); reactions are strided over the group's lanes; per-group LDS holds the
// concentrations, the species thermo, the per-reaction rate data and, while
// the Jacobian is assembled, the concentration Jacobian d wdot / d C.
#pragma once

#include <hip/hip_runtime.h>

#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "radau_core.hpp"

namespace acc {

constexpr int kKinMaxReactions = 4096;
// incidence-list entries fetched per LDS round trip in dydt, and in the
// Jacobian's d wdot / d C accumulation
constexpr int kKinRhsBatch = 8;
constexpr int kKinJacBatch = 8;
// Reactions a lane evaluates side by side in dydt.  A 64-lane group has the
// registers (one wave per SIMD) and no other wave to fill the waits: two at a
// time take the 54-state FP32-factor launch (65536 conditions) from 165.3 to
// 162.1 ms.  16-lane groups run two waves per SIMD on half the registers: two at a
// time spill (262144 14-state conditions, FP64: 30.0 -> 37.7 ms).
constexpr int rxn_unroll(int G) { return G == 64 ? 2 : 1; }

// *p += v in LDS, no return value: the LDS applies a wavefront's operations
// in issue order, so successive adds to one address keep their order.
__device__ __forceinline__ void lds_add(double* p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
constexpr double kKinR = 8.31446261815324;
constexpr double kKinPatm = 101325.0;
constexpr double kKinLnTref = 6.907755278982137;  // ln(1000)
constexpr double kKinLnC0R = -4.407418589020958;   // ln(1e-6 * 101325 / R): ln C0 = this - ln T
// Guards that keep f finite for any finite state: Newton trial states of a
// violent transient can carry T <= 0 or T ~ 1e7 K (ln T undefined, exp
// overflow) or mass fractions whose weighted sums vanish, and the Radau error
// norm maps NaN to its 1e-10 floor (fmax), i.e. would accept such a state.
// Physical trajectories never come near the guards.
constexpr double kKinTmin = 200.0;
constexpr double kKinTmax = 1.0e4;
constexpr double kKinSmin = 1.0e-3;
constexpr double kKinCpmin = 1.0;

// One reaction as the rate loop reads it, from global memory (each lane only
// its own reactions): rate parameters, net mole change, and the byte offsets of
// its six slots' species in the group's (C, g/RT) pairs -- reactants 0..2,
// products 3..5, empty slots the dummy species NS (C = 1, g = h = 0), so the
// loop has no test per slot.
struct alignas(16) KinReaction {
  double lnA, beta, EaR, dnu;
  uint16_t off[6];
  uint16_t pad[2];
};
static_assert(sizeof(KinReaction) == 48, "three 16-byte loads");

// Device view of a network: one packed blob (built by KineticsHost).  Its
// first lds_bytes (the tables that are read at data-dependent indices by the
// Jacobian) are copied by every block into the front of its LDS at kernel
// start; what a lane reads only for its own species or reactions stays in
// global memory (cache resident).  Species tables carry the dummy species NS.
// Byte offsets:
//   [off_invW] double invW[ns + 1]  [off_sl] uint64 slots[nr] (byte a = species of slot a, ns = empty)
//   [off_co]   int csr_off[ns + 1]  [off_ce] int csr[nnz] = (reaction << 8) | (nu & 0xff)
//   ---- end of the LDS part (lds_bytes) ----
//   [off_W]    double W[ns + 1]     [off_th] double thermo[5 (ns + 1)]
//   [off_rx]   KinReaction[nr]
//   [off_el]   the incidence list once more, for dydt: ell_batches batches of
//              kKinRhsBatch entries for every species (int ell[batch][half][ns + 1][4]),
//              entry = (byte offset of the reaction's q in the group's LDS << 16) | (nu & 0xffff);
//              lists end in entries that add 0 x 0
struct KinParams {
  const double* blob;  // device copy
  int blob_bytes;      // multiple of 16
  int lds_bytes;       // multiple of 16, the LDS-resident prefix
  int ns, nr, nnz;
  int off_invW, off_W, off_th, off_sl, off_co, off_ce, off_rx, off_el, ell_batches;
};

template <int NTOT>
struct MechKinetics {
  static constexpr int N = NTOT;
  static constexpr int NS = NTOT - 1;
  using Params = KinParams;
  static constexpr bool kJacInLds = true;
  // Networks above 64 states (a wavefront per condition, two rows per lane):
  // the parked Jacobian and the d wdot / d C rows do not fit the LDS; they live
  // in the group's global workspace, column-major with leading dimension
  // kJacLd, every row written and read only by the lane that owns it.
  static constexpr bool kLarge = NTOT > 64;
  static constexpr bool kJacColMajor = kLarge;
  static constexpr int kJacLd = kLarge ? 128 : NTOT;
  static_assert(!kLarge || NTOT <= 128, "networks of at most 128 states");
  // doubles of global workspace per group (0: none)
  __host__ __device__ static constexpr size_t global_doubles() {
    return kLarge ? (size_t)kJacLd * N + (size_t)kJacLd * NS : 0;
  }

  // Callbacks: dydt returns the rows a lane owns; jacob writes the dense
  // Jacobian into the group's LDS (kJacInLds), where the integrator keeps it.
  //
  // per group: (C, gRT) pairs, hR, cpR [NS + 1 each]; kf, kr, q, qT [nr each]; the
  // Jacobian buffer [N*N] (d wdot / d C rows while the Jacobian is assembled,
  // then the parked Jacobian).
  __host__ __device__ static size_t group_doubles(int nr) {
    return (size_t)4 * (NS + 1) + (size_t)4 * nr + (kLarge ? 0 : (size_t)N * N);
  }
  static size_t lds_bytes(const Params& p, int groups) {
    return (size_t)p.lds_bytes + groups * group_doubles(p.nr) * sizeof(double);
  }

  // Whole block: copy the network tables into LDS (before any divergence).
  __device__ __forceinline__ static void block_init(const Params& p, double* lds) {
    const int n16 = p.lds_bytes / 16;
    const int4* src = reinterpret_cast<const int4*>(p.blob);
    int4* dst = reinterpret_cast<int4*>(lds);
    for (int i = threadIdx.x; i < n16; i += blockDim.x) dst[i] = src[i];
    __syncthreads();
  }

  struct Ctx {
    int nr, ell_batches;
    const double* invW;
    const double* W;
    const double* thermo;
    const KinReaction* rx;
    const int4* ell;
    const unsigned long long* slots;
    const int* csr_off;
    const int* csr;
    double2* cg;  // (C, g/RT) per species
    double* hR;
    double* cpR;
    double* kf;
    double* kr;
    double* q;
    double* qT;
    double* Jc;
    double* jac;
    // tables copied by block_init at `lds`; group g's buffers after them
    __device__ Ctx(const Params& pp, int g, double* lds)
        : Ctx(pp, lds, lds + pp.lds_bytes / 8 + (size_t)g * group_doubles(pp.nr)) {}
    // tables at `tables`, the group's buffers at `group` (group_doubles(nr) doubles)
    __device__ Ctx(const Params& pp, const double* tables, double* group)
        : nr(pp.nr), ell_batches(pp.ell_batches) {
      const char* t = reinterpret_cast<const char*>(tables);
      const char* gl = reinterpret_cast<const char*>(pp.blob);
      invW = reinterpret_cast<const double*>(t + pp.off_invW);
      W = reinterpret_cast<const double*>(gl + pp.off_W);
      thermo = reinterpret_cast<const double*>(gl + pp.off_th);
      rx = reinterpret_cast<const KinReaction*>(gl + pp.off_rx);
      ell = reinterpret_cast<const int4*>(gl + pp.off_el);
      slots = reinterpret_cast<const unsigned long long*>(t + pp.off_sl);
      csr_off = reinterpret_cast<const int*>(t + pp.off_co);
      csr = reinterpret_cast<const int*>(t + pp.off_ce);
      double* b = group;
      cg = reinterpret_cast<double2*>(b); b += 2 * (NS + 1);
      hR = b; b += NS + 1;
      cpR = b; b += NS + 1;
      kf = b; b += pp.nr;
      kr = b; b += pp.nr;
      q = b; b += pp.nr;
      qT = b; b += pp.nr;
      // d wdot / d C is fully consumed (column sums) before the caller parks
      // the Jacobian rows, so the two share one buffer
      if constexpr (kLarge) {
        Jc = jac = nullptr;  // bind_global
      } else {
        Jc = b;
        jac = b;
      }
    }
    // large networks: the parked Jacobian (kJacLd x N) and the d wdot / d C
    // rows (kJacLd x NS) in the group's global workspace (global_doubles())
    __device__ void bind_global(double* ws) {
      jac = ws;
      Jc = ws + (size_t)kJacLd * N;
    }
  };

  struct Mix {
    double T, lnT, iT, S, Ctot, cpm, dcpm;
  };

  // species of row q of this lane; rows that hold none (the temperature row,
  // padding rows) take the dummy species, so that no step below is conditional
  template <int G>
  __device__ __forceinline__ static int species(int q) {
    const int r = Grp<G>::lane() + G * q;
    return r >= 1 && r < N ? r - 1 : NS;
  }

  // Shared prologue: T, thermo of owned species (to LDS), mixture sums and
  // concentrations (to LDS).
  template <int G, int R, bool JAC>
  __device__ __forceinline__ static void prologue(Ctx& c, double P, const double (&y)[R], Mix& m) {
    double a0[R], a1[R], a2[R], bh[R], bs[R], iw[R], yv[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int s = species<G>(q);
      const double* a = c.thermo + 5 * s;
      a0[q] = a[0];
      a1[q] = a[1];
      a2[q] = a[2];
      bh[q] = a[3];
      bs[q] = a[4];
      iw[q] = c.invW[s];
      yv[q] = s < NS ? y[q] : 0.0;
    }
    const double T = fmin(fmax(Grp<G>::bcast(y[0], 0), kKinTmin), kKinTmax);
    const double lnT = log(T);
    const double iT = 1.0 / T;
    double Sp = 0.0, cpp = 0.0, dcp = 0.0;
    double g[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int s = species<G>(q);
      const double cp = a0[q] + a1[q] * T + a2[q] * T * T;
      const double h = a0[q] * T + a1[q] * T * T * 0.5 + a2[q] * T * T * T * (1.0 / 3.0) + bh[q];
      const double sR = a0[q] * lnT + a1[q] * T + a2[q] * T * T * 0.5 + bs[q];
      if (JAC) c.cpR[s] = cp;
      c.hR[s] = h;
      g[q] = h * iT - sR;
      Sp += yv[q] * iw[q];
      cpp += yv[q] * cp * iw[q];
      dcp += yv[q] * (a1[q] + 2 * a2[q] * T) * iw[q];
    }
    m.T = T;
    m.lnT = lnT;
    m.iT = iT;
    Grp<G>::sum2(Sp, cpp);
    m.S = fmax(Sp, kKinSmin);
    m.cpm = fmax(kKinR * cpp, kKinCpmin);
    m.dcpm = JAC ? kKinR * Grp<G>::sum(dcp) : 0.0;
    m.Ctot = (1e-6 / kKinR) * P * iT;
    const double cs = m.Ctot / m.S;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int s = species<G>(q);
      c.cg[s] = double2{s < NS ? cs * (yv[q] * iw[q]) : 1.0, g[q]};
    }
    group_lds_sync();
  }

  // Rate constants and rates of progress of the reactions this lane handles,
  // U at a time (independent chains through the exponentials and the gathers
  // of each other); the records of the next U are fetched one pass ahead.
  // Passes beyond nr repeat the last reaction.  Bound by issue and by the
  // exponentials' dependent chains; the dummy species and the precomputed
  // offsets took a pass from ~160 to ~90 instructions.
  template <int G, bool JAC, int U>
  __device__ __forceinline__ static void reactions(Ctx& c, const Mix& m) {
    const int ln = Grp<G>::lane();
    const double lnC0 = kKinLnC0R - m.lnT;  // ln(1e-6 P_atm / (R T))
    const double lnTr = m.lnT - kKinLnTref;
    const double iT = m.iT;
    const int last = c.nr - 1;
    const char* cg = reinterpret_cast<const char*>(c.cg);
    KinReaction nx[U];
#pragma unroll
    for (int u = 0; u < U; ++u) nx[u] = c.rx[min(ln + u * G, last)];
#pragma unroll 1
    for (int j0 = 0; j0 < c.nr; j0 += U * G) {
      KinReaction x[U];
      double2 v[U][6];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = nx[u];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int a = 0; a < 6; ++a) v[u][a] = *reinterpret_cast<const double2*>(cg + x[u].off[a]);
      if (j0 + U * G < c.nr) {
#pragma unroll
        for (int u = 0; u < U; ++u) nx[u] = c.rx[min(j0 + ln + (U + u) * G, last)];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = min(j0 + ln + u * G, last);
        const double sum_nu_g = 0.0 - v[u][0].y - v[u][1].y - v[u][2].y + v[u][3].y + v[u][4].y + v[u][5].y;
        double pf = v[u][0].x * v[u][1].x * v[u][2].x;
        double pr = v[u][3].x * v[u][4].x * v[u][5].x;
        const double lnkf = x[u].lnA + x[u].beta * lnTr - x[u].EaR * iT;
        const double lnKc = -sum_nu_g + x[u].dnu * lnC0;
        const double kf = exp(lnkf);
        const double kr = exp(lnkf - lnKc);
        pf *= kf;
        pr *= kr;
        c.q[j] = pf - pr;
        if (JAC) {
          double h[6];
#pragma unroll
          for (int a = 0; a < 6; ++a) h[a] = c.hR[x[u].off[a] / 16];
          const double sum_nu_h = 0.0 - h[0] - h[1] - h[2] + h[3] + h[4] + h[5];
          const double dlnkf = (x[u].beta + x[u].EaR * iT) * iT;
          const double dlnkr = dlnkf - (sum_nu_h * iT - x[u].dnu) * iT;
          c.qT[j] = pf * dlnkf - pr * dlnkr;
          c.kf[j] = kf;
          c.kr[j] = kr;
        }
      }
    }
    group_lds_sync();
  }

  // Bound at one wave per SIMD by issue and exposed LDS round trips.  Without
  // per-slot tests, with the species' lists read from global memory as whole
  // batches (5 instead of 13 instructions per entry) and with nothing
  // conditional, states bit-identical: 32768 54-state conditions of one global
  // step FP64 117.1 -> 106.7 ms, 65536 with FP32 factors 185.3 -> 162.1 ms, 262144
  // 14-state conditions of two steps 35.2 -> 30.0 ms.
  template <int G, int R>
  __device__ __forceinline__ static void dydt(Ctx& c, double, double P, const double (&y)[R],
                                              double (&f)[R]) {
    const int ln = Grp<G>::lane();
    Mix m;
    prologue<G, R, false>(c, P, y, m);
    reactions<G, false, rxn_unroll(G)>(c, m);
    const double D = m.S / m.Ctot;
    const char* base = reinterpret_cast<const char*>(c.cg);
    double Qp = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      // incidence list in batches of eight, all lists as long as the longest:
      // the batch after this one is fetched while this one's rates are summed
      // in list order; entries beyond a list's end add an exact zero
      const int s = species<G>(q);
      const int4* e = c.ell + s;
      int4 n0 = e[0], n1 = e[NS + 1];
      double w = 0.0;
#pragma unroll 1
      for (int b = 0; b < c.ell_batches; ++b) {
        const int ce[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
        double qv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) qv[i] = *reinterpret_cast<const double*>(base + ((unsigned)ce[i] >> 16));
        if (b + 1 < c.ell_batches) {
          e += 2 * (NS + 1);
          n0 = e[0];
          n1 = e[NS + 1];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) w += (double)(short)ce[i] * qv[i];
      }
      f[q] = s < NS ? c.W[s] * w * D : 0.0;
      Qp += c.hR[s] * w;
    }
    const double Q = kKinR * Grp<G>::sum(Qp);
    const double fT = -Q * D / m.cpm;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (ln + G * q == 0) f[q] = fT;
    group_lds_sync();  // LDS is reused by the next evaluation
  }

  // Dense Jacobian, written as rows into the group's parked-Jacobian buffer:
  // c.jac[r*N + j] = d f_r / d y_j (row 0 = T).  The buffer doubles as the
  // d wdot / d C scratch, so each lane keeps its own d wdot / d C row in
  // registers until every lane has finished reading the scratch.  JB:
  // incidence-list entries per batch (the caller's choice: only a 64-lane group
  // with FP32 factors has the registers; FP64 factors fill the register file,
  // and 16-lane groups run two waves per SIMD on half of it).
  static constexpr int kJacBatchFP32 = kKinJacBatch;
  static constexpr int kJacBatchFP64 = 1;
  template <int G, int R, int JB = kKinJacBatch>
  __device__ __forceinline__ static void jacob(Ctx& c, double t, double P, const double (&y)[R]) {
    if constexpr (kLarge) {
      jacob_large<G, R>(c, P, y);
      return;
    }
    const int ln = Grp<G>::lane();
    Mix m;
    prologue<G, R, true>(c, P, y, m);
    reactions<G, true, 1>(c, m);
    const double S = m.S, Ctot = m.Ctot, iT = m.iT;
    const double D = S / Ctot;
    double Qp = 0.0, dQp = 0.0;
    double jr[R][NS];
    double rsv[R], wv[R], wTv[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
      rsv[q] = wv[q] = wTv[q] = 0.0;
#pragma unroll
      for (int i = 0; i < NS; ++i) jr[q][i] = 0.0;
      if (r >= 1 && r < N) {
        const int s = r - 1;
        double* row = c.Jc + (size_t)s * NS;
#pragma unroll
        for (int i = 0; i < NS; ++i) row[i] = 0.0;
        double w = 0.0, wT = 0.0;
        const int e1 = c.csr_off[s + 1];
        // incidence list in batches: the batch's entries, their reaction
        // data and the concentrations those reactions read are fetched
        // before any is used; the row updates are LDS atomic adds without
        // return, which a wavefront's LDS applies in issue order -- the
        // same sums in the same order as load-add-store, without a round
        // trip per update
        constexpr int B = JB;
#pragma unroll 1
        for (int e = c.csr_off[s]; e < e1; e += B) {
          int ce[B];
          double qv[B], qTv[B], kfv[B], krv[B];
          unsigned long long swv[B];
#pragma unroll
          for (int i = 0; i < B; ++i) ce[i] = c.csr[min(e + i, e1 - 1)];
#pragma unroll
          for (int i = 0; i < B; ++i) {
            const int j = ce[i] >> 8;
            qv[i] = c.q[j];
            qTv[i] = c.qT[j];
            kfv[i] = c.kf[j];
            krv[i] = c.kr[j];
            swv[i] = c.slots[j];
          }
          double cv[B][6];
#pragma unroll
          for (int i = 0; i < B; ++i)
#pragma unroll
            for (int a = 0; a < 6; ++a) {
              const int sa = (int)((swv[i] >> (8 * a)) & 0xffu);
              cv[i][a] = c.cg[sa].x;  // 1 for an empty slot
            }
#pragma unroll
          for (int i = 0; i < B; ++i) {
            if (e + i < e1) {
              const double nu = (double)(signed char)(ce[i] & 0xff);
              w += nu * qv[i];
              wT += nu * qTv[i];
              const double kfj = nu * kfv[i], krj = -nu * krv[i];
#pragma unroll
              for (int b = 0; b < 6; ++b) {
                const int sb = (int)((swv[i] >> (8 * b)) & 0xffu);
                if (sb != NS) {
                  double v = b < 3 ? kfj : krj;
                  const int lo = b < 3 ? 0 : 3;
#pragma unroll
                  for (int a = lo; a < lo + 3; ++a)
                    if (a != b) v *= cv[i][a];
                  lds_add(&row[sb], v);
                }
              }
            }
          }
        }
        // own row into registers; r_s = sum_m Jc[s][m] C_m
        double rs = 0.0;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
          jr[q][i] = row[i];
          rs += jr[q][i] * c.cg[i].x;
        }
        rsv[q] = rs;
        wv[q] = w;
        wTv[q] = wT;
        const double hs = c.hR[s];
#pragma unroll
        for (int i = 0; i < NS; ++i) row[i] = hs * (Ctot * jr[q][i] - rs);
        Qp += hs * w;
        dQp += c.cpR[s] * w + hs * (wT - rs * iT);
      }
    }
    const double Q = kKinR * Grp<G>::sum(Qp);
    const double dQdT = kKinR * Grp<G>::sum(dQp);
    group_lds_sync();
    // column sums of the H-weighted species rows: the lane owning row i+1 sums
    // column i (sixteen loads per round trip, summed in row order) and forms
    // entry i+1 of the temperature row from it -- the row's 53 entries in
    // parallel rather than one lane's loop of divisions
    const double cpm = m.cpm;
    const double QD = Q * D;
    double trow[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
      trow[q] = 0.0;
      if (r >= 1 && r < N) {
        const int i = r - 1;
        double sum = 0.0;
#pragma unroll 16
        for (int k = 0; k < NS; ++k) sum += c.Jc[(size_t)k * NS + i];
        const double iw = c.invW[i];
        const double dQdYi = kKinR * sum * iw / S;
        trow[q] = -(D * dQdYi + Q * iw / Ctot) / cpm + QD * kKinR * c.cpR[i] * iw / (cpm * cpm);
      }
    }
    group_lds_sync();  // the scratch is dead from here on: rows go to c.jac
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
      if (r == 0) {
        c.jac[0] = -(D * dQdT + QD * iT) / cpm + QD * m.dcpm / (cpm * cpm);
      } else if (r < N) {
        c.jac[r] = trow[q];  // temperature row, column r
        const int s = r - 1;
        const double Ws = c.W[s];
        const double corr = (rsv[q] - wv[q]) / Ctot;
        double* out = c.jac + (size_t)r * N;
#pragma unroll
        for (int i = 0; i < NS; ++i) out[1 + i] = Ws * c.invW[i] * (jr[q][i] - corr);
        out[0] = Ws * D * (wTv[q] + (wv[q] - rsv[q]) * iT);
      }
    }
    group_lds_sync();
  }

  // The same Jacobian for large networks: each lane accumulates its own rows
  // of d wdot / d C in the global workspace (element (r, i) at r + i kJacLd),
  // the temperature row's column sums of the H-weighted rows are group
  // reductions, and the parked Jacobian goes to the workspace column-major.
  template <int G, int R>
  __device__ static void jacob_large(Ctx& c, double P, const double (&y)[R]) {
    constexpr int LD = kJacLd;
    const int ln = Grp<G>::lane();
    Mix m;
    prologue<G, R, true>(c, P, y, m);
    reactions<G, true, 1>(c, m);
    const double S = m.S, Ctot = m.Ctot, iT = m.iT;
    const double D = S / Ctot;
    double Qp = 0.0, dQp = 0.0, HRp = 0.0;
    double rsv[R], wv[R], wTv[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
      rsv[q] = wv[q] = wTv[q] = 0.0;
      if (r >= 1 && r < N) {
        const int s = r - 1;
        double* row = c.Jc + r;
#pragma unroll 4
        for (int i = 0; i < NS; ++i) row[(size_t)i * LD] = 0.0;
        double w = 0.0, wT = 0.0;
        const int e1 = c.csr_off[s + 1];
#pragma unroll 1
        for (int e = c.csr_off[s]; e < e1; ++e) {
          const int ce = c.csr[e];
          const int j = ce >> 8;
          const double nu = (double)(signed char)(ce & 0xff);
          w += nu * c.q[j];
          wT += nu * c.qT[j];
          const unsigned long long sw = c.slots[j];
          int sp[6];
          double cv[6];
#pragma unroll
          for (int a = 0; a < 6; ++a) {
            sp[a] = (int)((sw >> (8 * a)) & 0xffu);
            cv[a] = c.cg[sp[a]].x;  // 1 for an empty slot
          }
          const double kfj = nu * c.kf[j], krj = -nu * c.kr[j];
#pragma unroll
          for (int b = 0; b < 6; ++b) {
            if (sp[b] != NS) {
              double v = b < 3 ? kfj : krj;
              const int lo = b < 3 ? 0 : 3;
#pragma unroll
              for (int a = lo; a < lo + 3; ++a)
                if (a != b) v *= cv[a];
              row[(size_t)sp[b] * LD] += v;
            }
          }
        }
        double rs = 0.0;
#pragma unroll 4
        for (int i = 0; i < NS; ++i) rs += row[(size_t)i * LD] * c.cg[i].x;
        rsv[q] = rs;
        wv[q] = w;
        wTv[q] = wT;
        const double hs = c.hR[s];
        Qp += hs * w;
        dQp += c.cpR[s] * w + hs * (wT - rs * iT);
        HRp += hs * rs;
      }
    }
    const double Q = kKinR * Grp<G>::sum(Qp);
    const double dQdT = kKinR * Grp<G>::sum(dQp);
    const double HR = Grp<G>::sum(HRp);
    const double cpm = m.cpm, QD = Q * D;
    // temperature row (owned by lane 0): column i of the H-weighted rows
#pragma unroll 1
    for (int i = 0; i < NS; ++i) {
      double part = 0.0;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = ln + G * q;
        if (r >= 1 && r < N) part += c.hR[r - 1] * c.Jc[r + (size_t)i * LD];
      }
      const double col = Ctot * Grp<G>::sum(part) - HR;
      if (ln == 0) {
        const double iw = c.invW[i];
        const double dQdYi = kKinR * col * iw / S;
        c.jac[(size_t)(1 + i) * LD] = -(D * dQdYi + Q * iw / Ctot) / cpm + QD * kKinR * c.cpR[i] * iw / (cpm * cpm);
      }
    }
    if (ln == 0) c.jac[0] = -(D * dQdT + QD * iT) / cpm + QD * m.dcpm / (cpm * cpm);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
      if (r >= 1 && r < N) {
        const int s = r - 1;
        const double Ws = c.W[s];
        const double corr = (rsv[q] - wv[q]) / Ctot;
        const double* jr = c.Jc + r;
        double* out = c.jac + r;
#pragma unroll 4
        for (int i = 0; i < NS; ++i) out[(size_t)(1 + i) * LD] = Ws * c.invW[i] * (jr[(size_t)i * LD] - corr);
        out[0] = Ws * D * (wTv[q] + (wv[q] - rsv[q]) * iT);
      }
    }
    group_lds_sync();  // LDS is reused by the next evaluation
  }
};

using MechKinetics14 = MechKinetics<14>;
using MechKinetics54 = MechKinetics<54>;
using MechKinetics112 = MechKinetics<112>;

// Host-side owner of a kinetics network: validation, the species -> reaction
// incidence list, and the device copies.
struct KineticsHost {
  int ns = 0, nr = 0;
  std::vector<double> W, invW, thermo, rc;
  std::vector<int> slots, csr_off, csr_rxn, csr_nu;
  void* dmem = nullptr;
  KinParams dev{};

  bool set(int ns_, int nr_, const double* W_, const double* th, const int* sl, const double* lnA,
           const double* beta, const double* EaR, std::string* msg) {
    if (ns_ <= 0 || nr_ <= 0 || !W_ || !th || !sl || !lnA || !beta || !EaR) {
      *msg = "accelerInt_set_kinetics: bad arguments";
      return false;
    }
    for (int s = 0; s < ns_; ++s)
      if (!(W_[s] > 0)) {
        *msg = "accelerInt_set_kinetics: molecular weights must be positive";
        return false;
      }
    for (int k = 0; k < 6 * nr_; ++k)
      if (sl[k] < -1 || sl[k] >= ns_) {
        *msg = "accelerInt_set_kinetics: slot species index out of range";
        return false;
      }
    ns = ns_;
    nr = nr_;
    W.assign(W_, W_ + ns);
    invW.resize(ns);
    for (int s = 0; s < ns; ++s) invW[s] = 1.0 / W[s];
    thermo.assign(th, th + 5 * ns);
    slots.assign(sl, sl + 6 * nr);
    rc.resize(3 * nr);
    for (int j = 0; j < nr; ++j) {
      rc[3 * j] = lnA[j];
      rc[3 * j + 1] = beta[j];
      rc[3 * j + 2] = EaR[j];
    }
    // net stoichiometric coefficients nu[s][j], kept in reaction order
    csr_off.assign(ns + 1, 0);
    csr_rxn.clear();
    csr_nu.clear();
    std::vector<std::vector<std::pair<int, int>>> lists(ns);
    for (int j = 0; j < nr; ++j) {
      int nu[6] = {0};
      int spc[6];
      int m = 0;
      for (int a = 0; a < 6; ++a) {
        const int s = slots[6 * j + a];
        if (s < 0) continue;
        int idx = -1;
        for (int b = 0; b < m; ++b)
          if (spc[b] == s) idx = b;
        if (idx < 0) {
          idx = m++;
          spc[idx] = s;
        }
        nu[idx] += a < 3 ? -1 : 1;
      }
      for (int b = 0; b < m; ++b)
        if (nu[b] != 0) lists[spc[b]].push_back({j, nu[b]});
    }
    for (int s = 0; s < ns; ++s) {
      csr_off[s + 1] = csr_off[s] + (int)lists[s].size();
      for (auto& e : lists[s]) {
        csr_rxn.push_back(e.first);
        csr_nu.push_back(e.second);
      }
    }
    return true;
  }

  bool upload(std::string* msg) {
    release();
    // packed blob, every section 16-byte aligned (see KinParams)
    const int nnz = (int)csr_rxn.size();
    std::vector<char> blob;
    auto section = [&](const void* src, size_t bytes) {
      const int off = (int)blob.size();
      blob.resize(blob.size() + ((bytes + 15) / 16) * 16, 0);
      if (bytes) memcpy(blob.data() + off, src, bytes);
      return off;
    };
    std::vector<unsigned long long> sl(nr);
    for (int j = 0; j < nr; ++j) {
      unsigned long long w = 0;
      for (int a = 0; a < 6; ++a) {
        const int sp = slots[6 * j + a];
        w |= (unsigned long long)(sp < 0 ? ns : sp) << (8 * a);
      }
      sl[j] = w;
    }
    std::vector<int> ce(nnz > 0 ? nnz : 1, 0);
    for (int e = 0; e < nnz; ++e) ce[e] = (csr_rxn[e] << 8) | (csr_nu[e] & 0xff);
    dev.ns = ns;
    dev.nr = nr;
    dev.nnz = nnz;
    // species tables with the dummy species (all zero) at the end
    std::vector<double> invWd(invW), Wd(W), thd(thermo);
    invWd.push_back(0.0);
    Wd.push_back(0.0);
    thd.resize(5 * ((size_t)ns + 1), 0.0);
    std::vector<KinReaction> rx(nr);
    for (int j = 0; j < nr; ++j) {
      KinReaction& r = rx[j];
      r = KinReaction{};
      r.lnA = rc[3 * j];
      r.beta = rc[3 * j + 1];
      r.EaR = rc[3 * j + 2];
      for (int a = 0; a < 6; ++a) {
        const int sp = slots[6 * j + a];
        if (sp >= 0) r.dnu += a < 3 ? -1.0 : 1.0;
        r.off[a] = (uint16_t)(16 * (sp < 0 ? ns : sp));
      }
    }
    // dydt's incidence list: every species as many whole batches as the longest
    static_assert(kKinRhsBatch == 8, "two int4 per batch");
    int longest = 0;
    for (int s = 0; s < ns; ++s) longest = std::max(longest, csr_off[s + 1] - csr_off[s]);
    dev.ell_batches = std::max(1, (longest + 7) / 8);
    const int zero = 8 * (3 * (ns + 1) - 1), q0 = 8 * (4 * (ns + 1) + 2 * nr);
    std::vector<int> el((size_t)dev.ell_batches * 2 * (ns + 1) * 4, (int)((unsigned)zero << 16));
    for (int s = 0; s < ns; ++s)
      for (int e = csr_off[s]; e < csr_off[s + 1]; ++e) {
        const int i = e - csr_off[s];
        el[(((size_t)(i / 4)) * (ns + 1) + s) * 4 + i % 4] =
            (int)(((unsigned)(q0 + 8 * csr_rxn[e]) << 16) | ((unsigned)csr_nu[e] & 0xffffu));
      }
    dev.off_invW = section(invWd.data(), invWd.size() * sizeof(double));
    dev.off_sl = section(sl.data(), (size_t)nr * sizeof(unsigned long long));
    dev.off_co = section(csr_off.data(), (size_t)(ns + 1) * sizeof(int));
    dev.off_ce = section(ce.data(), (size_t)ce.size() * sizeof(int));
    dev.lds_bytes = (int)blob.size();
    dev.off_W = section(Wd.data(), Wd.size() * sizeof(double));
    dev.off_th = section(thd.data(), thd.size() * sizeof(double));
    dev.off_rx = section(rx.data(), rx.size() * sizeof(KinReaction));
    dev.off_el = section(el.data(), el.size() * sizeof(int));
    dev.blob_bytes = (int)blob.size();
    if (hipMalloc(&dmem, blob.size()) != hipSuccess) {
      *msg = "hipMalloc failed for kinetics tables";
      dmem = nullptr;
      return false;
    }
    if (hipMemcpy(dmem, blob.data(), blob.size(), hipMemcpyHostToDevice) != hipSuccess) {
      *msg = "hipMemcpy failed for kinetics tables";
      return false;
    }
    dev.blob = (const double*)dmem;
    return true;
  }

  template <int NTOT>
  KinParams params() const {
    return dev;
  }

  void release() {
    if (dmem) hipFree(dmem);
    dmem = nullptr;
  }
};

}  // namespace acc
