// libaccelerint_hip.so: accelerInt-compatible C ABI over the gfx950 batched
// Radau IIA-5 kernels.
//
// Host side mirrors generic/solver_interface.cu:88-225 (initialize / integrate /
// cleanup), generic/solver_generic.cu:29-42 (one kernel launch per global step)
// and radau2a/radau2a_init.cu / radau2a_props.cu (solver hooks, check_error).
// Differences by design: the device layout is condition-major (y[c*N + i]),
// the transposition to and from the caller's column-major y_host happens on the
// device, and the per-condition workspace lives in registers/LDS instead of
// global memory, so required_solver_size() is the few bytes of per-condition
// HBM state.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <string>
#include <vector>

#include "accelerint.h"
#include "mech_fd.hpp"
#include "mech_kinetics.hpp"
#include "mech_vdp.hpp"
#include "radau_core.hpp"
#ifdef ACCELERINT_USER_MECHANISM
// A user-mechanism build (python -m accelerint_amd.build --mechanism DIR):
// the user's callbacks are the library's one mechanism, as the reference
// compiles one mechanism into each build; the built-in van der Pol and
// kinetics launches are left out of it.
#include "mech_user.hpp"
#define ACC_BUILTINS 0
#else
#define ACC_BUILTINS 1
#endif

// Waves per SIMD the register allocator targets (defaults; van der Pol and
// the 14-state network also have the autotuner's alternatives, kShapes*).
#ifndef ACC_VDP_WPE
#define ACC_VDP_WPE 2
#endif
#ifndef ACC_K14_WPE
#define ACC_K14_WPE 2
#endif
#ifndef ACC_K54_WPE
#define ACC_K54_WPE 1
#endif

namespace acc {

constexpr int kBlock = 256;

// The integration kernel: the analogue of the reference's per-step intDriver
// launch (solver_generic.cu:29-42) wrapped in its host global-step loop
// (solver_interface.cu:234-274), turned inside out.  Conditions are
// independent, so one launch runs every global step of a condition back to
// back; lane groups are persistent and pull condition indices from an atomic
// work counter.  A group advances one step attempt per loop iteration, so the
// moment its condition (or global step) ends it starts the next one -- no
// group idles waiting for a slow neighbour and no grid-wide barrier separates
// global steps.
template <int G>
__device__ __forceinline__ int grab_condition(int* work) {
  int c = 0;
  if (Grp<G>::lane() == 0) c = atomicAdd(work, 1);
  return Grp<G>::bcast_i(c, 0);
}

// The network's inference as a real call: its temporaries (MFMA tiles,
// activations) then never compete with the integrator's long-lived registers
// for the hot loop's allocation; the call's register save/restore happens
// once per global step.
struct MlpStages {
  double z1, z2, z3;
};
template <int N>
__device__ __attribute__((noinline)) MlpStages mlp_predict_call(const MlpView& m, double yr, double logh,
                                                                double logp) {
  MlpStages r;
  mlp_predict_wave<N>(m, yr, logh, logp, r.z1, r.z2, r.z3);
  return r;
}

// Learned Newton start for the first step of a global step (one condition
// per wavefront; the network's system size must match).  A prediction with a
// non-finite component anywhere in the group is dropped (zero start), and a
// condition whose predicted start was once discarded (see Radau::StartFailed)
// gets none for the rest of the launch.
template <class Mech, int G, int R, class St>
__device__ __forceinline__ void predict_start(const SolverParams& P, double pr, St& st) {
  if constexpr (G == 64 && R == 1 && Mech::N + 2 <= 64) {
    if (P.mlp.on && P.mlp.n == Mech::N) {
      double z1[1], z2[1], z3[1];
      if (st.StartFailed) return;
      const MlpStages zs = mlp_predict_call<Mech::N>(P.mlp, st.y[0], log(st.H), log(pr));
      z1[0] = zs.z1;
      z2[0] = zs.z2;
      z3[0] = zs.z3;
      const bool bad = !(__builtin_isfinite(z1[0]) && __builtin_isfinite(z2[0]) && __builtin_isfinite(z3[0]));
      if (Grp<G>::sum(bad ? 1.0 : 0.0) == 0.0) st.set_start(z1, z2, z3);
    }
  }
}

// One batch of conditions of one mechanism, condition-major in HBM.
//
// Escalation (mixed precision): with `esc` set, a condition that ends with a
// non-zero code or a non-finite state is not written back; its index is
// appended to esc[1..] (esc[0] = count) for an FP64 pass, which runs the same
// code over that list (`list`, with its length read from `num_dev`) from the
// untouched initial state.
struct Queue {
  int num;
  const double* pr;
  double* y;
  int* codes;
  uint32_t* counters;
  int* work;
  const int* list;
  const int* num_dev;
  int* esc;
  float* cost;  // per-condition work of this call (queue ordering of the next)
};

// Work of one condition over a call, in units of one right-hand-side
// evaluation: the relative costs of the events on the 54-state network
// (LU pair ~12 dydt, Jacobian ~8, a Newton or error-estimate solve ~1).
__device__ __forceinline__ float work_estimate(const uint32_t (&cnt)[NCNT]) {
  return (float)cnt[CNT_F] + 12.0f * (float)cnt[CNT_LU] + 8.0f * (float)cnt[CNT_JAC] +
         (float)(cnt[CNT_NEWTON] + cnt[CNT_ES]);
}

// Global workspace of a group (large systems): the memory-resident factors
// first (MemLU layout, rounded to 256 B), then the mechanism's buffers.
template <class M, class = void>
struct MechGlobal : std::integral_constant<size_t, 0> {};
template <class M>
struct MechGlobal<M, std::void_t<decltype(M::global_doubles())>>
    : std::integral_constant<size_t, M::global_doubles()> {};

template <class Mech, int G, int R, class MT>
constexpr size_t factor_ws_bytes() {
  using St = Radau<Mech, G, R, MT>;
  return St::kMemLU ? ((St::MLU::bytes() + 255) / 256) * 256 : 0;
}
// bytes per group, the same for both precisions (sized for FP64 factors)
template <class Mech, int G, int R>
constexpr size_t group_ws_bytes() {
  return factor_ws_bytes<Mech, G, R, double>() + MechGlobal<Mech>::value * sizeof(double);
}

// The group's slice of P.ws (null when the kernel needs none).
__device__ __forceinline__ char* group_ws(const SolverParams& P, size_t group) {
  return P.ws ? P.ws + group * P.ws_bytes : nullptr;
}

// The persistent loop of a lane group over a queue: pull a condition, run all
// of its global steps back to back (one step attempt per iteration), write it
// back, pull the next.  LS: the learned Newton start is compiled in (a
// separate instantiation, so the network's inference code adds no register
// pressure to runs without it).
template <class Mech, int G, int R, class MT, bool LS = false>
__device__ __forceinline__ void run_queue(const Queue& qa, double t_start, double t_end, double step,
                                          const SolverParams& P, typename Mech::Ctx& ctx, double* zs = nullptr,
                                          char* gws = nullptr) {
  constexpr int N = Mech::N;
  const int ln = Grp<G>::lane();
  const int num = qa.num_dev ? *qa.num_dev : qa.num;
  Radau<Mech, G, R, MT> st;
  st.zs = zs;
  if constexpr (Radau<Mech, G, R, MT>::kMemLU) st.ws = reinterpret_cast<MT*>(gws);
  if constexpr (MechGlobal<Mech>::value > 0)
    ctx.bind_global(reinterpret_cast<double*>(gws + factor_ws_bytes<Mech, G, R, double>()));
  uint32_t cnt[NCNT];
  double prc = 0.0, t_next = t_end;
  int k = 0;
  int ci = grab_condition<G>(qa.work);
  int c = 0;
  bool fresh = true;
#pragma unroll 1
  while (ci < num) {
    if (fresh) {  // load condition c and open its first global step
      c = qa.list ? qa.list[ci] : ci;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = ln + G * q;
        st.y[q] = (r < N) ? qa.y[(size_t)c * N + r] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < NCNT; ++i) cnt[i] = 0;
      prc = qa.pr[c];
      st.StartFailed = false;
      k = 0;
      t_next = fmin(t_end, t_start + step);
      st.begin(P, t_start, t_next);
      if constexpr (LS) predict_start<Mech, G, R>(P, prc, st);
      fresh = false;
    }
    int code = EC_success;
    if (!st.finished()) code = st.attempt(ctx, P, prc, cnt);
    if (code == RADAU_CONTINUE) continue;
    if (code == EC_success && t_next + kRoundoff < t_end) {  // next global step
      const double t0 = t_next;
      ++k;
      t_next = fmin(t_end, t_start + (k + 1) * step);
      st.begin(P, t0, t_next);
      if constexpr (LS) predict_start<Mech, G, R>(P, prc, st);
      continue;
    }
    // condition finished (all steps done, or an error code): write back, or
    // hand it to the FP64 pass
    bool escalate = false;
    if (qa.esc) {
      double bad = 0.0;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (ln + G * q < N && !isfinite(st.y[q])) bad = 1.0;
      escalate = code != EC_success || Grp<G>::sum(bad) != 0.0;
    }
    if (!escalate) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = ln + G * q;
        if (r < N) qa.y[(size_t)c * N + r] = st.y[q];
      }
    }
    if (ln == 0) {
      if (escalate) qa.esc[1 + atomicAdd(qa.esc, 1)] = c;
      else if (qa.codes) qa.codes[c] = code;
      if (qa.counters) {
#pragma unroll
        for (int i = 0; i < NCNT; ++i) qa.counters[(size_t)c * NCNT + i] += cnt[i];
      }
      if (qa.cost) qa.cost[c] = work_estimate(cnt);
    }
    ci = grab_condition<G>(qa.work);
    fresh = true;
  }
}

template <class Mech, int G, int R, int BLOCK, int WPE, class MT, bool LS = false>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void k_radau(
    Queue qa, double t_start, double t_end, double step, SolverParams P, typename Mech::Params mp, int start_off,
    int groups) {
  extern __shared__ double lds_dyn[];
  // the group index, wave-uniform when a group is a whole wavefront: read
  // into a scalar register so the group's LDS and workspace addresses stay
  // out of the vector register file
  const int g = G == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / G) : (int)(threadIdx.x / G);
  Mech::block_init(mp, lds_dyn);
  typename Mech::Ctx ctx(mp, g, lds_dyn);
  // learned start: the group's predicted stages after the mechanism's LDS
  double* zs = LS ? lds_dyn + start_off + (size_t)g * 3 * G * R : nullptr;
  char* gws = group_ws(P, (size_t)blockIdx.x * (BLOCK / G) + g);
  if constexpr (G > 1) {
    // the block's working groups: one per wavefront, then a second one per
    // wavefront, and so on (no block barrier follows)
    constexpr int kWaveGroups = 64 / G;
    if ((g % kWaveGroups) * (BLOCK / 64) + g / kWaveGroups >= groups) return;
  }
  run_queue<Mech, G, R, MT, LS>(qa, t_start, t_end, step, P, ctx, zs, gws);
}

// Heterogeneous batch in one persistent launch: the 112-, 54- and 14-state
// networks.  Every wavefront drains the 112-state queue (one condition per
// wave, factors and Jacobian in its global workspace), then the 54-state queue
// (one condition per wave), then the 14-state queue (four 16-lane groups per
// wave), so the long jobs start first.  LDS: the 54- and 14-state networks'
// tables (the 112-state tables are read from global memory here), then one
// region per wave that serves each size's group buffers in turn.
template <class MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_radau_hetero(
    Queue q112, Queue q54, Queue q14, double t_start, double t_end, double step, SolverParams P, KinParams mp112,
    KinParams mp54, KinParams mp14, int off14, int off_regions, int region_doubles) {
  extern __shared__ double lds_dyn[];
  MechKinetics54::block_init(mp54, lds_dyn);
  MechKinetics14::block_init(mp14, lds_dyn + off14);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);  // wave-uniform (scalar register)
  double* region = lds_dyn + off_regions + (size_t)w * region_doubles;
  if (q112.num > 0) {
    // a wave per 112-state condition; its tables stay in global memory (L2)
    MechKinetics112::Ctx ctx(mp112, mp112.blob, region);
    run_queue<MechKinetics112, 64, 2, MT>(q112, t_start, t_end, step, P, ctx, nullptr,
                                          group_ws(P, (size_t)blockIdx.x * 4 + w));
  }
  {
    MechKinetics54::Ctx ctx(mp54, lds_dyn, region);
    run_queue<MechKinetics54, 64, 1, MT>(q54, t_start, t_end, step, P, ctx);
  }
  {
    const int g = (threadIdx.x & 63) / 16;
    MechKinetics14::Ctx ctx(mp14, lds_dyn + off14, region + (size_t)g * MechKinetics14::group_doubles(mp14.nr));
    run_queue<MechKinetics14, 16, 1, MT>(q14, t_start, t_end, step, P, ctx);
  }
}

__global__ void k_iota(int* out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = i;
}

__global__ void k_reset_work(int* work, int* esc) {
  *work = 0;
  if (esc) *esc = 0;
}

// Evaluates the mechanism callbacks at every condition's state (no
// integration): dy[c*N + i] and jac[c*N*N + i + j*N] (column-major per
// condition).  Counterpart of the reference's rate/Jacobian dump test
// (tests/rateOutputTest.cu:18).
template <class Mech, int G, int R, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_eval_callbacks(int num, double t,
                                                          const double* __restrict__ pr,
                                                          const double* __restrict__ y,
                                                          double* __restrict__ dy,
                                                          double* __restrict__ jac,
                                                          typename Mech::Params mp, char* gws) {
  extern __shared__ double lds_dyn[];
  constexpr int N = Mech::N;
  constexpr int GPB = BLOCK / G;
  const int g = threadIdx.x / G;
  const int c = blockIdx.x * GPB + g;
  Mech::block_init(mp, lds_dyn);
  if (c >= num) return;
  const int ln = threadIdx.x % G;
  double yl[R], f[R], J[R][N];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = ln + G * q;
    yl[q] = (r < N) ? y[(size_t)c * N + r] : 0.0;
  }
  typename Mech::Ctx ctx(mp, g, lds_dyn);
  if constexpr (MechGlobal<Mech>::value > 0)  // a workspace slice per condition
    ctx.bind_global(reinterpret_cast<double*>(gws) + (size_t)c * MechGlobal<Mech>::value);
  Mech::template dydt<G, R>(ctx, t, pr[c], yl, f);
  if constexpr (Mech::kJacInLds) {
    Mech::template jacob<G, R>(ctx, t, pr[c], yl);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int r = ln + G * q;
#pragma unroll
      for (int j = 0; j < N; ++j) J[q][j] = (r < N) ? ctx.jac[jidx<Mech>(r, j)] : 0.0;
    }
  } else {
    Mech::template jacob<G, R>(ctx, t, pr[c], yl, J);
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = ln + G * q;
    if (r < N) {
      dy[(size_t)c * N + r] = f[q];
#pragma unroll
      for (int j = 0; j < N; ++j) jac[(size_t)c * N * N + r + (size_t)j * N] = J[q][j];
    }
  }
}

// Kernels whose dynamic LDS exceeds 64 KiB declare it before launch.
template <class K>
hipError_t allow_lds(K kern, size_t lds) {
  if (lds <= 65536) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)lds);
}

template <class Mech, int G, int R, int BLOCK>
hipError_t launch_eval(int num, double t, const double* pr, const double* y, double* dy,
                       double* jac, const typename Mech::Params& mp, hipStream_t s, char* gws = nullptr) {
  constexpr int GPB = BLOCK / G;
  const int blocks = (num + GPB - 1) / GPB;
  if (blocks == 0) return hipSuccess;
  auto kern = k_eval_callbacks<Mech, G, R, BLOCK>;
  const size_t lds = Mech::lds_bytes(mp, GPB);
  hipError_t e = allow_lds(kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(BLOCK), lds, s, num, t, pr, y, dy, jac, mp, gws);
  return hipGetLastError();
}

// Column-major (i*ld + c) <-> condition-major (c*n + i) transposition.
__global__ void k_cm_to_cond(const double* __restrict__ src, double* __restrict__ dst, int num,
                             int n, int ld) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)num * n) return;
  const int c = (int)(idx / n), i = (int)(idx % n);
  dst[idx] = src[(size_t)i * ld + c];
}
__global__ void k_cond_to_cm(const double* __restrict__ src, double* __restrict__ dst, int num,
                             int n, int ld) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)num * n) return;
  const int c = (int)(idx % num), i = (int)(idx / num);
  dst[(size_t)i * ld + c] = src[(size_t)c * n + i];
}

// Why the last launch was refused before reaching the device (empty if none).
std::string g_launch_msg;

// Persistent grid: as many blocks as fit on the device at once (capped by the
// number of conditions).  The group's LDS share must fit the device's
// per-block limit and leave at least one resident block per CU.
template <class Mech, int G, int R, int BLOCK, int WPE, class MT, bool LS = false>
hipError_t launch_radau(int num, double t_start, double t_end, double step, const double* pr,
                        double* y, int* codes, uint32_t* cnt, int* work, const int* list,
                        const int* num_dev, int* esc, const SolverParams& P,
                        const typename Mech::Params& mp, hipStream_t s, float* cost = nullptr) {
  constexpr int GPB = BLOCK / G;
  auto kern = k_radau<Mech, G, R, BLOCK, WPE, MT, LS>;
  const size_t lds_mech = Mech::lds_bytes(mp, GPB);
  // learned start: 3 stages x R rows x G lanes of doubles per group after the mechanism's share
  const size_t lds = lds_mech + (LS ? (size_t)GPB * 3 * G * R * sizeof(double) : 0);
  static int resident = 0;     // blocks per device that fit at once, per instantiation
  static size_t lds_ok = 0;    // LDS size the residency was computed for
  if (resident == 0 || lds_ok != lds) {
    int dev = 0, cus = 0, per_cu = 0, max_lds = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    if (lds > (size_t)max_lds) {
      char buf[256];
      snprintf(buf, sizeof buf, "k_radau needs %zu B of LDS per block (%d lane groups), device allows %d",
               lds, GPB, max_lds);
      g_launch_msg = buf;
      return hipErrorInvalidConfiguration;
    }
    e = allow_lds(kern, lds);
    if (e != hipSuccess) return e;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, BLOCK, lds);
    if (e != hipSuccess) return e;
    if (per_cu <= 0) {
      g_launch_msg = "k_radau: no block fits on a compute unit";
      return hipErrorInvalidConfiguration;
    }
    resident = (cus > 0 ? cus : 1) * per_cu;
    lds_ok = lds;
  }
  if (num <= 0) return hipSuccess;  // (num = 0: only the occupancy queries above)
  // Working groups per block.  A batch that does not fill the device is spread
  // over all of it: groups that share a wavefront run each other's branches and
  // iterations, and wavefronts that share a CU its instruction cache (16-lane
  // groups, FP64 ignition: 100 conditions 5.18 -> 4.60 ms, 1000 4.79 -> 4.13 ms;
  // 64-lane groups, 33 conditions 81.6 -> 80.0 ms).  From one condition per
  // resident group on, all of them work.  One-lane groups fill their wavefronts
  // as before: 300 conditions gained (1.26 -> 1.10 ms), 5000 did not (1.44 ->
  // 1.45 ms) and 262144, where no group is left out, lost (0.54 -> 0.60 ms) by
  // the test alone.
  int groups = G > 1 ? (num - 1) / resident + 1 : GPB;
  if (groups > GPB) groups = GPB;
  int blocks = (num - 1) / groups + 1;
  if (blocks > resident) blocks = resident;
  if constexpr (group_ws_bytes<Mech, G, R>() > 0) {
    // a global workspace slice per group: no more groups than slices
    if (!P.ws || P.ws_bytes < group_ws_bytes<Mech, G, R>() || P.ws_groups < GPB) {
      g_launch_msg = "k_radau: the large-system workspace is missing (install the network before initialize)";
      return hipErrorInvalidValue;
    }
    if (blocks * GPB > P.ws_groups) {
      blocks = P.ws_groups / GPB;
      groups = GPB;
    }
  }
  hipLaunchKernelGGL(k_reset_work, dim3(1), dim3(1), 0, s, work, esc);
  const Queue qa{num, pr, y, codes, cnt, work, list, num_dev, esc, cost};
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(BLOCK), lds, s, qa, t_start, t_end, step, P, mp,
                     (int)(lds_mech / sizeof(double)), groups);
  return hipGetLastError();
}

// factor_test.hip: the row LU on caller matrices (orders 2, 14, 54).
hipError_t launch_factor_test(int n, bool fp32, bool cplx, int num, const double* are, const double* aim,
                              const double* bre, const double* bim, double* lre, double* lim, int* perm, int* info,
                              double* xre, double* xim, char* ws, hipStream_t s);
size_t factor_test_ws_bytes(int n);

}  // namespace acc

using namespace acc;

// Device memory of accelerInt_integrate_device_noalloc, the entry point that
// allocates nothing: [0] the persistent queue's work counter, [1] the count of
// conditions the FP32-factor pass hands to the FP64 pass, [2 ..] their
// indices.  Every GPU the library runs on holds one copy (1 MiB) until the
// process ends; host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (g_noalloc_scratch).
constexpr int kNoAllocMaxConditions = 262144;
static __device__ __align__(256) int scratch[2 + kNoAllocMaxConditions];

// ---- library state (one context per process, like solver_interface.cu:17-28) ---
namespace {

constexpr int kMaxDevices = 64;
int* g_noalloc_scratch[kMaxDevices] = {};  // device address of `scratch`, per device

struct State {
#if ACC_BUILTINS
  int mech = ACCELERINT_MECH_VAN_DER_POL;
  int n = 2;
#else
  int mech = ACCELERINT_MECH_USER;
  int n = kUserN;
#endif
  int precision = ACCELERINT_PRECISION_FP64;
  int jacobian = ACCELERINT_JACOBIAN_ANALYTIC;
  int fd_order = 1;  // finite-difference order of the FD Jacobian (FD_ORD)
  int learned = 0;          // learned Newton start on (the network is looked up per launch)
  float* own_log_x = nullptr;  // library-owned training-sample log (accelerInt_start_log)
  float* own_log_z = nullptr;
  int* own_log_n = nullptr;
  int own_log_cap = 0;
  hipGraph_t graph = nullptr;          // captured integration (accelerInt_graph_capture)
  hipGraphExec_t graph_exec = nullptr;
  int* graph_order = nullptr;          // the captured launch's queue order (owned by the graph)
  int graph_order_num = 0;
  int graph_mlp_gen = -1;              // start-network generation the graph reads (-1: zero start)
  SolverParams P{1e-10, 1e-6, 0};
  int abort_on_error = 1;
  int device = -1;
  int padded = 0;     // capacity in conditions of the device buffers
  hipStream_t stream = nullptr;
  double* d_y = nullptr;    // condition-major state
  double* d_ycm = nullptr;  // column-major staging for host transfers
  double* d_pr = nullptr;
  int* d_codes = nullptr;
  uint32_t* d_cnt = nullptr;
  int* d_work = nullptr;    // atomic work counter of the persistent kernel
  int* d_work2 = nullptr;   // second queue of a heterogeneous launch
  int* d_esc2 = nullptr;    // escalation list of the second queue
  int* d_esc = nullptr;     // escalation list of the mixed-precision pass: [count, indices...]
  // queue order (longest first by the previous call's measured work)
  int schedule = ACCELERINT_SCHEDULE_LONGEST_FIRST;
  float* d_cost = nullptr;     // per-condition work of the last call
  uint32_t* d_keys = nullptr;  // sorted keys (radix-sort output, unused)
  int* d_iota = nullptr;
  int* d_order = nullptr;      // condition indices, most work first
  void* d_sort_tmp = nullptr;
  size_t sort_tmp_bytes = 0;
  int cost_num = 0;   // conditions d_cost describes (0: none)
  int order_num = 0;  // conditions d_order is a permutation of (0: none)
  bool capturing = false;
  bool chunked = false;
  std::vector<int> h_codes;
  int have_status = 0;
  // kinetics tables (device copies)
  // one kinetics network per compiled size (14 and 54 states); kin_n = the
  // size of the primary one (the most recently installed)
  KineticsHost kin14, kin54, kin112;
  int kin_n = 0;
  MechKinetics14::Params kp14{};
  MechKinetics54::Params kp54{};
  MechKinetics112::Params kp112{};
  // global workspace of the 112-state kernels (memory-resident factors and
  // parked Jacobian), ws_groups groups of ws_bytes
  char* d_ws = nullptr;
  size_t ws_bytes = 0;
  int ws_groups = 0;
  int* d_work3 = nullptr;  // third queue of a heterogeneous launch
  int* d_esc3 = nullptr;
  std::string err;
  // launch shapes (waves per SIMD) by [system: 0 vdP, 1 14-state][precision]
  int wpe[2][2] = {{ACC_VDP_WPE, ACC_VDP_WPE}, {ACC_K14_WPE, ACC_K14_WPE}};
} S;

// Launch shapes the autotuner chooses among: waves per SIMD the register
// allocator targets (512 / WPE registers per lane; fewer waves, fewer spills).
// The 54-state kernel has one shape: four 54-state groups fill the LDS of a
// CU and need all 512 registers of a lane, so one wave per SIMD.
constexpr int kShapesVdp[] = {1, 2, 4};
constexpr int kShapesK14[] = {1, 2, 3};

static_assert(kShapesVdp[1] == ACC_VDP_WPE && kShapesK14[1] == ACC_K14_WPE, "defaults are the middle shapes");

int shape_system() { return S.mech == ACCELERINT_MECH_VAN_DER_POL ? 0 : (S.n == 14 ? 1 : -1); }

std::string device_key() {
  hipDeviceProp_t prop;
  if (S.device < 0 || hipGetDeviceProperties(&prop, S.device) != hipSuccess) return "";
  char buf[300];
  snprintf(buf, sizeof buf, "%s/%dCU", prop.gcnArchName, prop.multiProcessorCount);
  for (char* c = buf; *c; ++c)
    if (*c == '"' || *c == '\\') *c = '_';
  return buf;
}

// Tuning cache: a JSON array with one object per line,
//   {"device": "...", "n_states": N, "precision": P, "waves_per_simd": W, "ms": [...]}
// Lines of other devices, sizes or precisions are kept as they are.
struct TuneEntry {
  std::string device;
  int n = 0, precision = 0, wpe = 0;
  std::string line;
};

std::vector<TuneEntry> read_tuning(const char* path) {
  std::vector<TuneEntry> out;
  FILE* fp = fopen(path, "r");
  if (!fp) return out;
  char buf[2048];
  while (fgets(buf, sizeof buf, fp)) {
    TuneEntry e;
    char dev[512];
    const char* p = strstr(buf, "{\"device\": \"");
    if (!p || sscanf(p, "{\"device\": \"%511[^\"]\", \"n_states\": %d, \"precision\": %d, \"waves_per_simd\": %d",
                     dev, &e.n, &e.precision, &e.wpe) != 4)
      continue;
    e.device = dev;
    e.line = p;
    while (!e.line.empty() && (e.line.back() == '\n' || e.line.back() == ',' || e.line.back() == ' ' ||
                               e.line.back() == ']'))
      e.line.pop_back();
    out.push_back(e);
  }
  fclose(fp);
  return out;
}

bool write_tuning(const char* path, const std::vector<TuneEntry>& entries) {
  const std::string tmp = std::string(path) + ".tmp";
  FILE* fp = fopen(tmp.c_str(), "w");
  if (!fp) return false;
  fprintf(fp, "[\n");
  for (size_t i = 0; i < entries.size(); ++i)
    fprintf(fp, "%s%s\n", entries[i].line.c_str(), i + 1 < entries.size() ? "," : "");
  fprintf(fp, "]\n");
  if (fclose(fp) != 0) return false;
  return rename(tmp.c_str(), path) == 0;
}

void set_err(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  S.err = buf;
}

// gpuAssert analogue (examples/van_der_pol/gpu_macros.cuh:26-34): record the
// error; in abort mode print it and exit with the HIP error code.
bool hip_ok(hipError_t e, const char* what) {
  if (e == hipSuccess) return true;
  set_err("HIP error in %s: %s", what, hipGetErrorString(e));
  if (S.abort_on_error) {
    fprintf(stderr, "GPUassert: %s %s\n", hipGetErrorString(e), what);
    exit((int)e);
  }
  return false;
}
#define HIPOK(x) hip_ok((x), #x)

size_t bytes_per_condition() {
  // y (condition-major) + staging copy + parameter + code + escalation slot + counters
  return (size_t)S.n * sizeof(double) * 2 + sizeof(double) + 2 * sizeof(int) + NCNT * sizeof(uint32_t);
}

void free_buffers() {
  if (S.d_y) hipFree(S.d_y);
  if (S.d_ycm) hipFree(S.d_ycm);
  if (S.d_pr) hipFree(S.d_pr);
  if (S.d_codes) hipFree(S.d_codes);
  if (S.d_cnt) hipFree(S.d_cnt);
  if (S.d_work) hipFree(S.d_work);
  if (S.d_esc) hipFree(S.d_esc);
  if (S.d_work2) hipFree(S.d_work2);
  if (S.d_esc2) hipFree(S.d_esc2);
  if (S.d_work3) hipFree(S.d_work3);
  if (S.d_esc3) hipFree(S.d_esc3);
  if (S.d_ws) hipFree(S.d_ws);
  S.d_work3 = S.d_esc3 = nullptr;
  S.d_ws = nullptr;
  S.ws_bytes = 0;
  S.ws_groups = 0;
  S.P.ws = nullptr;
  S.P.ws_bytes = 0;
  S.P.ws_groups = 0;
  if (S.d_cost) hipFree(S.d_cost);
  if (S.d_keys) hipFree(S.d_keys);
  if (S.d_iota) hipFree(S.d_iota);
  if (S.d_order) hipFree(S.d_order);
  if (S.d_sort_tmp) hipFree(S.d_sort_tmp);
  S.d_cost = nullptr;
  S.d_keys = nullptr;
  S.d_iota = S.d_order = nullptr;
  S.d_sort_tmp = nullptr;
  S.sort_tmp_bytes = 0;
  S.cost_num = S.order_num = 0;
  S.d_work2 = nullptr;
  S.d_esc2 = nullptr;
  S.d_work = nullptr;
  S.d_esc = nullptr;
  S.d_y = S.d_ycm = S.d_pr = nullptr;
  S.d_codes = nullptr;
  S.d_cnt = nullptr;
  S.padded = 0;
}

bool alloc_buffers(int cap) {
  free_buffers();
  if (!HIPOK(hipMalloc(&S.d_y, (size_t)cap * S.n * sizeof(double)))) return false;
  if (!HIPOK(hipMalloc(&S.d_ycm, (size_t)cap * S.n * sizeof(double)))) return false;
  if (!HIPOK(hipMalloc(&S.d_pr, (size_t)cap * sizeof(double)))) return false;
  if (!HIPOK(hipMalloc(&S.d_codes, (size_t)cap * sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_cnt, (size_t)cap * NCNT * sizeof(uint32_t)))) return false;
  if (!HIPOK(hipMemset(S.d_cnt, 0, (size_t)cap * NCNT * sizeof(uint32_t)))) return false;
  if (!HIPOK(hipMalloc(&S.d_work, sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_esc, ((size_t)cap + 1) * sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_work2, sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_esc2, ((size_t)cap + 1) * sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_work3, sizeof(int)))) return false;
  if (!HIPOK(hipMalloc(&S.d_esc3, ((size_t)cap + 1) * sizeof(int)))) return false;
  if (S.kin112.ns == 111) {
    // one 256-thread block (four 112-state groups) per compute unit: the
    // kernels' LDS (tables and group buffers) leaves room for no second one
    int dev = 0, cus = 0;
    if (!HIPOK(hipGetDevice(&dev)) ||
        !HIPOK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)))
      return false;
    S.ws_groups = 4 * (cus > 0 ? cus : 1);
    S.ws_bytes = group_ws_bytes<MechKinetics112, 64, 2>();
    if (!HIPOK(hipMalloc(&S.d_ws, S.ws_bytes * (size_t)S.ws_groups))) return false;
    S.P.ws = S.d_ws;
    S.P.ws_bytes = S.ws_bytes;
    S.P.ws_groups = S.ws_groups;
  }
  if (cap > 0) {
    if (!HIPOK(hipMalloc(&S.d_cost, (size_t)cap * sizeof(float)))) return false;
    if (!HIPOK(hipMalloc(&S.d_keys, (size_t)cap * sizeof(uint32_t)))) return false;
    if (!HIPOK(hipMalloc(&S.d_iota, (size_t)cap * sizeof(int)))) return false;
    if (!HIPOK(hipMalloc(&S.d_order, (size_t)cap * sizeof(int)))) return false;
    hipLaunchKernelGGL(k_iota, dim3((cap + 255) / 256), dim3(256), 0, 0, S.d_iota, cap);
    if (!HIPOK(hipGetLastError())) return false;
    if (!HIPOK(hipcub::DeviceRadixSort::SortPairsDescending(nullptr, S.sort_tmp_bytes, (const uint32_t*)S.d_cost,
                                                             S.d_keys, S.d_iota, S.d_order, cap)))
      return false;
    if (!HIPOK(hipMalloc(&S.d_sort_tmp, S.sort_tmp_bytes > 0 ? S.sort_tmp_bytes : 1))) return false;
  }
  S.padded = cap;
  S.h_codes.assign(cap, 0);
  return true;
}

// Lane-group shape per system size: van der Pol one condition per lane (two
// rows each); 14 states a 16-lane group (four conditions per wave); 54 states
// a whole wave per condition, four waves per block sharing the LDS tables.
template <class MT>
hipError_t launch_mt(int num, double t_start, double t_end, double step, const double* pr, double* y,
                     int* codes, uint32_t* cnt, const int* list, const int* num_dev, int* esc,
                     hipStream_t s, float* cost = nullptr, int* work = nullptr) {
  constexpr int prec = std::is_same<MT, float>::value ? 1 : 0;
  int* const wk = work ? work : S.d_work;  // the persistent queue's work counter
#if !ACC_BUILTINS
  (void)prec;
  if (S.mech != ACCELERINT_MECH_USER) return hipErrorInvalidValue;
  if (S.jacobian == ACCELERINT_JACOBIAN_FINITE_DIFFERENCE || !kUserHasJacobian)
    return launch_radau<MechFD<MechUser>, kUserG, kUserR, kUserBlock, kUserG == 64 ? 1 : 2, MT>(
        num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P,
        MechFD<MechUser>::Params{MechUser::Params{}, S.P.atol, S.P.rtol, S.fd_order}, s, cost);
  return launch_radau<MechUser, kUserG, kUserR, kUserBlock, kUserG == 64 ? 1 : 2, MT>(
      num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P, MechUser::Params{}, s, cost);
#else
  if (S.jacobian == ACCELERINT_JACOBIAN_FINITE_DIFFERENCE) {
    // finite-difference Jacobian: van der Pol and the 14- and 54-state networks
    // (the learned start is not compiled into these kernels)
    if (S.mech == ACCELERINT_MECH_VAN_DER_POL)
      return launch_radau<MechFD<MechVdP>, 1, 2, 256, ACC_VDP_WPE, MT>(
          num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P,
          MechFD<MechVdP>::Params{MechVdP::Params{}, S.P.atol, S.P.rtol, S.fd_order}, s, cost);
    if (S.mech == ACCELERINT_MECH_KINETICS && S.n == 14)
      return launch_radau<MechFD<MechKinetics14>, 16, 1, 128, ACC_K14_WPE, MT>(
          num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P,
          MechFD<MechKinetics14>::Params{S.kp14, S.P.atol, S.P.rtol, S.fd_order}, s, cost);
    if (S.mech == ACCELERINT_MECH_KINETICS && S.n == 54)
      return launch_radau<MechFD<MechKinetics54>, 64, 1, 256, ACC_K54_WPE, MT>(
          num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P,
          MechFD<MechKinetics54>::Params{S.kp54, S.P.atol, S.P.rtol, S.fd_order}, s, cost);
    g_launch_msg = "the finite-difference Jacobian is compiled for van der Pol and the 14- and 54-state networks";
    return hipErrorInvalidValue;
  }
  switch (S.mech) {
    case ACCELERINT_MECH_VAN_DER_POL: {
#define ACC_VDP_LAUNCH(W)                                                                                     \
  launch_radau<MechVdP, 1, 2, 256, W, MT>(num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, \
                                          esc, S.P, MechVdP::Params{}, s, cost)
      const int w = S.wpe[0][prec];
      if (w == kShapesVdp[0]) return ACC_VDP_LAUNCH(kShapesVdp[0]);
      if (w == kShapesVdp[2]) return ACC_VDP_LAUNCH(kShapesVdp[2]);
      return ACC_VDP_LAUNCH(kShapesVdp[1]);
#undef ACC_VDP_LAUNCH
    }
    case ACCELERINT_MECH_KINETICS:
      if (S.n == 14) {
#define ACC_K14_LAUNCH(W)                                                                                  \
  launch_radau<MechKinetics14, 16, 1, 128, W, MT>(num, t_start, t_end, step, pr, y, codes, cnt, wk, list, \
                                                  num_dev, esc, S.P, S.kp14, s, cost)
        const int w = S.wpe[1][prec];
        if (w == kShapesK14[0]) return ACC_K14_LAUNCH(kShapesK14[0]);
        if (w == kShapesK14[2]) return ACC_K14_LAUNCH(kShapesK14[2]);
        return ACC_K14_LAUNCH(kShapesK14[1]);
#undef ACC_K14_LAUNCH
      }
      if (S.n == 112)
        return launch_radau<MechKinetics112, 64, 2, 256, 1, MT>(num, t_start, t_end, step, pr, y, codes, cnt, wk,
                                                                 list, num_dev, esc, S.P, S.kp112, s, cost);
      if (S.n == 54 && S.learned)
        return launch_radau<MechKinetics54, 64, 1, 256, ACC_K54_WPE, MT, true>(
            num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P, S.kp54, s, cost);
      if (S.n == 54)
        return launch_radau<MechKinetics54, 64, 1, 256, ACC_K54_WPE, MT>(
            num, t_start, t_end, step, pr, y, codes, cnt, wk, list, num_dev, esc, S.P, S.kp54, s, cost);
      return hipErrorInvalidValue;
    default:
      return hipErrorInvalidValue;
  }
#endif
}

// Queue order of the next launch over num conditions: with the longest-first
// schedule and the previous call's per-condition work at hand (same number of
// conditions, one chunk), the condition indices sorted by that work,
// descending -- greedy list scheduling of the persistent groups then starts
// the expensive conditions first instead of meeting one at the end.  Inside a
// graph capture the sort is not recorded: the captured launch reads the
// graph's own copy of the order made before capture (later calls re-sort
// d_order for their own sizes, so the graph must not read it at replay).
// nullptr = index order.  Results do not depend on the order.
const int* queue_order(int num, hipStream_t s) {
  if (S.capturing) return S.graph_order_num == num ? S.graph_order : nullptr;
  if (S.schedule != ACCELERINT_SCHEDULE_LONGEST_FIRST || S.chunked || num < 2 || !S.d_order) return nullptr;
  if (!S.capturing && S.cost_num == num) {
    size_t bytes = S.sort_tmp_bytes;
    if (hipcub::DeviceRadixSort::SortPairsDescending(S.d_sort_tmp, bytes, (const uint32_t*)S.d_cost, S.d_keys,
                                                     S.d_iota, S.d_order, num, 0, 32, s) != hipSuccess)
      return nullptr;
    S.order_num = num;
  }
  return S.order_num == num ? S.d_order : nullptr;
}

// One integration of num <= S.padded conditions.  Mixed precision runs the
// FP32-factor kernel over all conditions, then the FP64 kernel over the
// conditions it escalated (the count stays on the device: no host sync).
// The learned start's network for this launch (S.P.mlp), or an error.
hipError_t prepare_start_network() {
  S.P.mlp = MlpView{};
  if (S.learned) {
    if (S.jacobian != ACCELERINT_JACOBIAN_ANALYTIC) {
      g_launch_msg = "the learned start is compiled with the analytic Jacobian only (turn one of them off)";
      return hipErrorInvalidValue;
    }
    if (S.n + 2 > 64) {
      g_launch_msg = "the learned start runs one condition per wavefront on N + 2 <= 64 features (N <= 62)";
      return hipErrorInvalidValue;
    }
    S.P.mlp = mlp_view();
    if (!S.P.mlp.on || S.P.mlp.n != S.n) {
      g_launch_msg = "learned start is on but no network for this system size is loaded";
      return hipErrorInvalidValue;
    }
  }
  return hipSuccess;
}

hipError_t launch(int num, double t_start, double t_end, double step, const double* pr, double* y,
                  int* codes, uint32_t* cnt, hipStream_t s) {
  g_launch_msg.clear();
  if (hipError_t e0 = prepare_start_network(); e0 != hipSuccess) return e0;
  if (num <= 0) {  // occupancy queries only
    hipError_t e = launch_mt<double>(0, t_start, t_end, step, pr, y, codes, cnt, nullptr, nullptr, nullptr, s);
    if (e == hipSuccess && S.precision == ACCELERINT_PRECISION_MIXED)
      e = launch_mt<float>(0, t_start, t_end, step, pr, y, codes, cnt, nullptr, nullptr, nullptr, s);
    return e;
  }
  const int* order = queue_order(num, s);
  float* cost = S.chunked ? nullptr : S.d_cost;
  hipError_t e;
  if (S.precision != ACCELERINT_PRECISION_MIXED) {
    e = launch_mt<double>(num, t_start, t_end, step, pr, y, codes, cnt, order, nullptr, nullptr, s, cost);
  } else {
    e = launch_mt<float>(num, t_start, t_end, step, pr, y, codes, cnt, order, nullptr, S.d_esc, s, cost);
    if (e == hipSuccess)
      e = launch_mt<double>(num, t_start, t_end, step, pr, y, codes, cnt, S.d_esc + 1, S.d_esc, nullptr, s, cost);
  }
  if (e == hipSuccess && cost) S.cost_num = num;
  return e;
}

// One integration with the queue's work counter and the escalation list in
// `sc` (the noalloc scratch): index order, no event counters, no cost record.
hipError_t launch_noalloc(int num, double t_start, double t_end, double step, const double* pr, double* y,
                          int* codes, int* sc, hipStream_t s) {
  g_launch_msg.clear();
  if (hipError_t e0 = prepare_start_network(); e0 != hipSuccess) return e0;
  if (S.precision != ACCELERINT_PRECISION_MIXED)
    return launch_mt<double>(num, t_start, t_end, step, pr, y, codes, nullptr, nullptr, nullptr, nullptr, s,
                             nullptr, sc);
  hipError_t e = launch_mt<float>(num, t_start, t_end, step, pr, y, codes, nullptr, nullptr, nullptr, sc + 1, s,
                                  nullptr, sc);
  if (e == hipSuccess)
    e = launch_mt<double>(num, t_start, t_end, step, pr, y, codes, nullptr, sc + 2, sc + 1, nullptr, s, nullptr,
                          sc);
  return e;
}

hipError_t launch_eval_any(int num, double t, const double* pr, const double* y, double* dy,
                           double* jac, hipStream_t s, char* gws) {
#if !ACC_BUILTINS
  if (S.mech == ACCELERINT_MECH_USER && kUserHasJacobian)
    return launch_eval<MechUser, kUserG, kUserR, kUserBlock>(num, t, pr, y, dy, jac, MechUser::Params{}, s);
  if (S.mech == ACCELERINT_MECH_USER)
    return launch_eval<MechFD<MechUser>, kUserG, kUserR, kUserBlock>(
        num, t, pr, y, dy, jac, MechFD<MechUser>::Params{MechUser::Params{}, S.P.atol, S.P.rtol, S.fd_order}, s);
  return hipErrorInvalidValue;
#else
  switch (S.mech) {
    case ACCELERINT_MECH_VAN_DER_POL:
      return launch_eval<MechVdP, 1, 2, 256>(num, t, pr, y, dy, jac, MechVdP::Params{}, s);
    case ACCELERINT_MECH_KINETICS:
      if (S.n == 14) return launch_eval<MechKinetics14, 16, 1, 128>(num, t, pr, y, dy, jac, S.kp14, s);
      if (S.n == 54) return launch_eval<MechKinetics54, 64, 1, 256>(num, t, pr, y, dy, jac, S.kp54, s);
      if (S.n == 112)
        return gws ? launch_eval<MechKinetics112, 64, 2, 256>(num, t, pr, y, dy, jac, S.kp112, s, gws)
                   : hipErrorInvalidValue;
      return hipErrorInvalidValue;
    default:
      return hipErrorInvalidValue;
  }
#endif
}

// Heterogeneous launch: the 14- and 54-state networks' batches in one
// persistent kernel; with mixed precision, then the FP64 passes over each
// batch's escalated conditions.
// P: the solver parameters of this launch (no sample log, no learned start:
// both are sized and trained for one network, and the two queues' records
// would interleave in one log).
template <class MT>
hipError_t launch_hetero(int n112, const double* pr112, double* y112, int* codes112, int n54, const double* pr54,
                         double* y54, int* codes54, int n14, const double* pr14, double* y14, int* codes14,
                         double t_start, double t_end, double step, const SolverParams& P, hipStream_t s) {
  constexpr bool kMixed = std::is_same<MT, float>::value;
  auto kern = k_radau_hetero<MT>;
  const int off14 = S.kp54.lds_bytes / 8;
  const int off_regions = off14 + S.kp14.lds_bytes / 8;
  const size_t r54 = MechKinetics54::group_doubles(S.kp54.nr);
  const size_t r14 = 4 * MechKinetics14::group_doubles(S.kp14.nr);
  const size_t r112 = n112 > 0 ? MechKinetics112::group_doubles(S.kp112.nr) : 0;
  size_t region_sz = r54 > r14 ? r54 : r14;
  region_sz = region_sz > r112 ? region_sz : r112;
  const int region = (int)region_sz;
  const size_t lds = ((size_t)off_regions + 4 * (size_t)region) * sizeof(double);
  static int resident = 0;
  static size_t lds_ok = 0;
  if (resident == 0 || lds_ok != lds) {
    int dev = 0, cus = 0, per_cu = 0, max_lds = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    if (lds > (size_t)max_lds) {
      char buf[200];
      snprintf(buf, sizeof buf, "heterogeneous launch needs %zu B of LDS per block, device allows %d", lds, max_lds);
      g_launch_msg = buf;
      return hipErrorInvalidConfiguration;
    }
    e = allow_lds(kern, lds);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 256, lds);
    if (e != hipSuccess) return e;
    if (per_cu <= 0) {
      g_launch_msg = "heterogeneous launch: no block fits on a compute unit";
      return hipErrorInvalidConfiguration;
    }
    resident = (cus > 0 ? cus : 1) * per_cu;
    lds_ok = lds;
  }
  int want = (n54 + 3) / 4 > (n14 + 15) / 16 ? (n54 + 3) / 4 : (n14 + 15) / 16;
  want = want > (n112 + 3) / 4 ? want : (n112 + 3) / 4;
  int blocks = want < resident ? want : resident;
  if (n112 > 0) {
    if (!P.ws || P.ws_groups < 4) {
      g_launch_msg = "heterogeneous launch: the 112-state workspace is missing (install the network before initialize)";
      return hipErrorInvalidValue;
    }
    if (blocks * 4 > P.ws_groups) blocks = P.ws_groups / 4;
  }
  if (blocks < 1) return hipSuccess;
  int* esc112 = kMixed ? S.d_esc3 : nullptr;
  int* esc54 = kMixed ? S.d_esc : nullptr;
  int* esc14 = kMixed ? S.d_esc2 : nullptr;
  hipLaunchKernelGGL(k_reset_work, dim3(1), dim3(1), 0, s, S.d_work3, esc112);
  hipLaunchKernelGGL(k_reset_work, dim3(1), dim3(1), 0, s, S.d_work, esc54);
  hipLaunchKernelGGL(k_reset_work, dim3(1), dim3(1), 0, s, S.d_work2, esc14);
  const Queue q112{n112, pr112, y112, codes112, nullptr, S.d_work3, nullptr, nullptr, esc112};
  const Queue q54{n54, pr54, y54, codes54, nullptr, S.d_work, nullptr, nullptr, esc54};
  const Queue q14{n14, pr14, y14, codes14, nullptr, S.d_work2, nullptr, nullptr, esc14};
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), lds, s, q112, q54, q14, t_start, t_end, step, P, S.kp112,
                     S.kp54, S.kp14, off14, off_regions, region);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !kMixed) return e;
  if (n112 > 0) {
    e = launch_radau<MechKinetics112, 64, 2, 256, 1, double>(n112, t_start, t_end, step, pr112, y112, codes112,
                                                              nullptr, S.d_work3, S.d_esc3 + 1, S.d_esc3, nullptr, P,
                                                              S.kp112, s);
    if (e != hipSuccess) return e;
  }
  if (n54 > 0) {
    e = launch_radau<MechKinetics54, 64, 1, 256, ACC_K54_WPE, double>(n54, t_start, t_end, step, pr54, y54, codes54,
                                                                      nullptr, S.d_work, S.d_esc + 1, S.d_esc,
                                                                      nullptr, P, S.kp54, s);
    if (e != hipSuccess) return e;
  }
  if (n14 > 0)
    e = launch_radau<MechKinetics14, 16, 1, 128, ACC_K14_WPE, double>(n14, t_start, t_end, step, pr14, y14, codes14,
                                                                      nullptr, S.d_work2, S.d_esc2 + 1, S.d_esc2,
                                                                      nullptr, P, S.kp14, s);
  return e;
}

// Global-step loop of solver_interface.cu:225-275 on device-resident,
// condition-major buffers: one launch covers every global step.
int run_steps(int num, double t_start, double t_end, double stepsize, double* y, const double* pr,
              int* codes, uint32_t* cnt, hipStream_t s) {
  const double step = stepsize < 0 ? t_end - t_start : stepsize;
  if (!(t_start + kRoundoff < t_end) || num <= 0) return 0;
  hipError_t e = hipSuccess;
  // chunks of at most `padded` conditions (the escalation list's capacity);
  // the queue ordering needs the whole batch in one chunk
  S.chunked = num > S.padded;
  if (S.chunked) S.cost_num = S.order_num = 0;
  for (int off = 0; off < num && e == hipSuccess; off += S.padded) {
    const int m = num - off < S.padded ? num - off : S.padded;
    e = launch(m, t_start, t_end, step, pr + off, y + (size_t)off * S.n, codes ? codes + off : nullptr,
               cnt ? cnt + (size_t)off * NCNT : nullptr, s);
  }
  if (e != hipSuccess && !g_launch_msg.empty()) {
    set_err("%s", g_launch_msg.c_str());
    if (S.abort_on_error) {
      fprintf(stderr, "%s\n", g_launch_msg.c_str());
      exit((int)e);
    }
    return -1;
  }
  return hip_ok(e, "k_radau launch") ? 0 : -1;
}

bool ensure_init() {
  if (S.device >= 0) return true;
  accelerInt_initialize(0, 0);
  return S.device >= 0;
}

}  // namespace

extern "C" {

int accelerInt_select_mechanism(int kind) {
  if (S.device >= 0) {
    set_err("accelerInt_select_mechanism must precede accelerInt_initialize");
    return -1;
  }
#if !ACC_BUILTINS
  if (kind == ACCELERINT_MECH_USER) return 0;
  set_err("this library is a user-mechanism build: its one mechanism is ACCELERINT_MECH_USER (%d states)", kUserN);
  return -1;
#endif
  if (kind == ACCELERINT_MECH_VAN_DER_POL) {
    S.mech = kind;
    S.n = 2;
    return 0;
  }
  if (kind == ACCELERINT_MECH_KINETICS) {
    if (S.kin_n == 0) {
      set_err("accelerInt_set_kinetics must be called before selecting the kinetics mechanism");
      return -1;
    }
    S.mech = kind;
    S.n = S.kin_n;
    return 0;
  }
  if (kind == ACCELERINT_MECH_USER) {
    set_err("this library carries no user mechanism (build one with python -m accelerint_amd.build --mechanism DIR)");
    return -1;
  }
  set_err("unknown mechanism kind %d", kind);
  return -1;
}

int accelerInt_set_kinetics(int ns, int nr, const double* W, const double* thermo, const int* slots,
                            const double* lnA, const double* beta, const double* EaR) {
  if (S.device >= 0) {
    set_err("accelerInt_set_kinetics must precede accelerInt_initialize");
    return -1;
  }
  if (!ACC_BUILTINS) {
    set_err("this library is a user-mechanism build: the built-in kinetics networks are not compiled into it");
    return -1;
  }
  if (ns + 1 != 14 && ns + 1 != 54 && ns + 1 != 112) {
    set_err("kinetics system size %d is not compiled (available: 14, 54, 112)", ns + 1);
    return -1;
  }
  if (nr <= 0 || nr > kKinMaxReactions) {
    set_err("kinetics reaction count %d out of range (1..%d)", nr, kKinMaxReactions);
    return -1;
  }
  std::string msg;
  KineticsHost& kin = (ns + 1 == 14) ? S.kin14 : (ns + 1 == 54 ? S.kin54 : S.kin112);
  if (!kin.set(ns, nr, W, thermo, slots, lnA, beta, EaR, &msg)) {
    set_err("%s", msg.c_str());
    return -1;
  }
  S.mech = ACCELERINT_MECH_KINETICS;
  S.n = ns + 1;
  S.kin_n = ns + 1;
  return 0;
}

// ---- files of the reference's command-line driver ---------------------------
// Initial conditions, generic/read_initial_conditions.c:30-78 with CONP: a
// binary file of NUM records of N + 2 doubles, [t, y_0, param, y_1 .. y_{N-1}]
// (y_0 = temperature, param = pressure for kinetics; the state needs no
// species mask: every species is part of it).
int accelerInt_read_initial_conditions(const char* filename, int NUM, double* y_host, double* var_host) {
  const int n = S.n;
  if (!filename || NUM <= 0 || !y_host || !var_host) {
    set_err("accelerInt_read_initial_conditions: bad arguments");
    return -1;
  }
  FILE* fp = fopen(filename, "rb");
  if (!fp) {
    set_err("Could not open file: %s", filename);
    return -1;
  }
  std::vector<double> rec((size_t)n + 2);
  for (int i = 0; i < NUM; ++i) {
    const size_t got = fread(rec.data(), sizeof(double), rec.size(), fp);
    if (got != rec.size()) {
      fclose(fp);
      set_err("File (%s) is incorrectly formatted: record %d has %zu of %d doubles", filename, i, got, n + 2);
      return -1;
    }
    y_host[i] = rec[1];
    var_host[i] = rec[2];
    for (int j = 1; j < n; ++j) y_host[i + (size_t)j * NUM] = rec[(size_t)j + 2];
  }
  fclose(fp);
  return 0;
}

// The reference's own entry point (generic/read_initial_conditions.h:12): it
// allocates the arrays and exits on a missing or short file.
void read_initial_conditions(const char* filename, int NUM, double** y_host, double** variable_host) {
  *y_host = (double*)malloc((size_t)NUM * S.n * sizeof(double));
  *variable_host = (double*)malloc((size_t)NUM * sizeof(double));
  if (!*y_host || !*variable_host ||
      accelerInt_read_initial_conditions(filename, NUM, *y_host, *variable_host) != 0) {
    fprintf(stderr, "%s\n", S.err.c_str());
    exit(-1);
  }
}

// State log of generic/solver_main.c:47-66 (write_log): the time, then N
// doubles per condition (y_0 .. y_{N-1}).  Appends unless append == 0.
int accelerInt_write_log(const char* path, int append, int NUM, double t, const double* y_host) {
  const int n = S.n;
  if (!path || NUM < 0 || (NUM > 0 && !y_host)) {
    set_err("accelerInt_write_log: bad arguments");
    return -1;
  }
  FILE* fp = fopen(path, append ? "ab" : "wb");
  if (!fp) {
    set_err("accelerInt_write_log: cannot open %s", path);
    return -1;
  }
  bool ok = fwrite(&t, sizeof(double), 1, fp) == 1;
  std::vector<double> rec(n);
  for (int c = 0; c < NUM && ok; ++c) {
    for (int i = 0; i < n; ++i) rec[i] = y_host[(size_t)i * NUM + c];
    ok = fwrite(rec.data(), sizeof(double), n, fp) == (size_t)n;
  }
  ok = (fclose(fp) == 0) && ok;
  if (!ok) set_err("accelerInt_write_log: write to %s failed", path);
  return ok ? 0 : -1;
}

// A kinetics network from a binary file: int32 ns, int32 nr, then W[ns],
// thermo[ns][5], slots int32[nr][6], lnA[nr], beta[nr], EaR[nr] (the arrays of
// accelerInt_set_kinetics, in that order).
int accelerInt_load_kinetics(const char* path) {
  FILE* fp = path ? fopen(path, "rb") : nullptr;
  if (!fp) {
    set_err("accelerInt_load_kinetics: cannot open %s", path ? path : "(null)");
    return -1;
  }
  int32_t hdr[2] = {0, 0};
  bool ok = fread(hdr, sizeof(int32_t), 2, fp) == 2 && hdr[0] > 0 && hdr[0] < 4096 && hdr[1] > 0 &&
            hdr[1] <= kKinMaxReactions;
  const int ns = hdr[0], nr = hdr[1];
  std::vector<double> W, th, lnA, beta, EaR;
  std::vector<int32_t> sl;
  if (ok) {
    W.resize(ns);
    th.resize((size_t)5 * ns);
    sl.resize((size_t)6 * nr);
    lnA.resize(nr);
    beta.resize(nr);
    EaR.resize(nr);
    ok = fread(W.data(), 8, W.size(), fp) == W.size() && fread(th.data(), 8, th.size(), fp) == th.size() &&
         fread(sl.data(), 4, sl.size(), fp) == sl.size() && fread(lnA.data(), 8, lnA.size(), fp) == lnA.size() &&
         fread(beta.data(), 8, beta.size(), fp) == beta.size() && fread(EaR.data(), 8, EaR.size(), fp) == EaR.size();
  }
  fclose(fp);
  if (!ok) {
    set_err("accelerInt_load_kinetics: %s is not a kinetics network file", path);
    return -1;
  }
  return accelerInt_set_kinetics(ns, nr, W.data(), th.data(), sl.data(), lnA.data(), beta.data(), EaR.data());
}

int accelerInt_set_tolerances(double atol, double rtol) {
  if (!(atol > 0) || !(rtol > 0)) {
    set_err("tolerances must be positive");
    return -1;
  }
  S.P.atol = atol;
  S.P.rtol = rtol;
  return 0;
}

int accelerInt_set_precision(int mode) {
  if (mode != ACCELERINT_PRECISION_FP64 && mode != ACCELERINT_PRECISION_MIXED) {
    set_err("unknown precision mode %d", mode);
    return -1;
  }
  S.precision = mode;
  return 0;
}

int accelerInt_set_jacobian(int mode) {
  if (mode != ACCELERINT_JACOBIAN_ANALYTIC && mode != ACCELERINT_JACOBIAN_FINITE_DIFFERENCE) {
    set_err("unknown Jacobian mode %d", mode);
    return -1;
  }
  S.jacobian = mode;
  return 0;
}

int accelerInt_set_fd_order(int order) {
  if (order != 1 && order != 2 && order != 4 && order != 6) {
    set_err("finite-difference order must be 1, 2, 4 or 6 (got %d)", order);
    return -1;
  }
  S.fd_order = order;
  return 0;
}

int accelerInt_set_schedule(int mode) {
  if (mode != ACCELERINT_SCHEDULE_INDEX && mode != ACCELERINT_SCHEDULE_LONGEST_FIRST) {
    set_err("unknown schedule mode %d", mode);
    return -1;
  }
  S.schedule = mode;
  return 0;
}

int accelerInt_get_schedule(float* work, int* order, int num) {
  if (S.device < 0) return -1;
  if (num < 0 || num > S.padded) {
    set_err("accelerInt_get_schedule: num must be 0..%d", S.padded);
    return -1;
  }
  if (!HIPOK(hipStreamSynchronize(S.stream))) return -1;
  const bool ready = S.schedule == ACCELERINT_SCHEDULE_LONGEST_FIRST && S.cost_num == num && num >= 2;
  if (ready) {  // the order the next call sorts to
    size_t bytes = S.sort_tmp_bytes;
    if (!HIPOK(hipcub::DeviceRadixSort::SortPairsDescending(S.d_sort_tmp, bytes, (const uint32_t*)S.d_cost,
                                                             S.d_keys, S.d_iota, S.d_order, num, 0, 32, S.stream)) ||
        !HIPOK(hipStreamSynchronize(S.stream)))
      return -1;
    S.order_num = num;
  }
  if (work && num > 0 && !HIPOK(hipMemcpy(work, S.d_cost, (size_t)num * sizeof(float), hipMemcpyDeviceToHost)))
    return -1;
  if (order && ready && !HIPOK(hipMemcpy(order, S.d_order, (size_t)num * sizeof(int), hipMemcpyDeviceToHost)))
    return -1;
  return ready ? num : 0;
}

int accelerInt_set_launch_shape(int n_states, int precision, int waves_per_simd) {
  const int sys = n_states == 2 ? 0 : (n_states == 14 ? 1 : -1);
  const int* shapes = sys == 0 ? kShapesVdp : kShapesK14;
  if (sys < 0 || (precision != 0 && precision != 1) ||
      (waves_per_simd != shapes[0] && waves_per_simd != shapes[1] && waves_per_simd != shapes[2])) {
    set_err("accelerInt_set_launch_shape: no shape with %d waves per SIMD for %d states", waves_per_simd, n_states);
    return -1;
  }
  S.wpe[sys][precision] = waves_per_simd;
  return 0;
}

int accelerInt_get_launch_shape(int n_states, int precision) {
  if (n_states == 54) return ACC_K54_WPE;
  const int sys = n_states == 2 ? 0 : (n_states == 14 ? 1 : -1);
  if (sys < 0 || (precision != 0 && precision != 1)) {
    set_err("accelerInt_get_launch_shape: unknown system size or precision");
    return -1;
  }
  return S.wpe[sys][precision];
}

// Times every launch shape of the selected system and precision on the given
// device-resident conditions (copied into the library's own state buffer, so
// y_dev is left untouched), keeps the fastest, and records it in cache_path
// (if given).  One untimed run per shape first, so module loading is not timed.
int accelerInt_autotune(int NUM, double t_start, double t_end, double stepsize, const double* y_dev,
                        const double* var_dev, const char* cache_path, double* ms_out) {
  if (!ensure_init()) return -1;
  if (NUM <= 0 || NUM > S.padded || !y_dev || !var_dev) {
    set_err("accelerInt_autotune: bad arguments (NUM must be 1..%d)", S.padded);
    return -1;
  }
  const int sys = shape_system();
  const int prec = S.precision == ACCELERINT_PRECISION_MIXED ? 1 : 0;
  if (sys < 0) return ACC_K54_WPE;  // a single shape
  const int* shapes = sys == 0 ? kShapesVdp : kShapesK14;
  const int keep = S.wpe[sys][prec];
  const size_t bytes = (size_t)NUM * S.n * sizeof(double);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (!HIPOK(hipEventCreate(&e0)) || !HIPOK(hipEventCreate(&e1))) return -1;
  double ms[3] = {0, 0, 0};
  int rc = 0;
  for (int k = 0; k < 3 && rc == 0; ++k) {
    S.wpe[sys][prec] = shapes[k];
    for (int pass = 0; pass < 2 && rc == 0; ++pass) {
      const int m = pass == 0 ? (NUM < 64 ? NUM : 64) : NUM;
      if (!HIPOK(hipMemcpyAsync(S.d_y, y_dev, bytes, hipMemcpyDeviceToDevice, S.stream)) ||
          !HIPOK(hipEventRecord(e0, S.stream))) {
        rc = -1;
        break;
      }
      rc = run_steps(m, t_start, t_end, stepsize, S.d_y, var_dev, S.d_codes, nullptr, S.stream);
      float t = 0.0f;
      if (rc == 0 && (!HIPOK(hipEventRecord(e1, S.stream)) || !HIPOK(hipEventSynchronize(e1)) ||
                      !HIPOK(hipEventElapsedTime(&t, e0, e1))))
        rc = -1;
      ms[k] = t;
    }
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  S.cost_num = S.order_num = 0;  // the timing runs' work does not describe the caller's next batch
  if (rc != 0) {
    S.wpe[sys][prec] = keep;
    return -1;
  }
  int best = 0;
  for (int k = 1; k < 3; ++k)
    if (ms[k] < ms[best]) best = k;
  S.wpe[sys][prec] = shapes[best];
  if (ms_out)
    for (int k = 0; k < 3; ++k) ms_out[k] = ms[k];
  if (cache_path) {
    std::vector<TuneEntry> entries = read_tuning(cache_path);
    const std::string dev = device_key();
    TuneEntry e;
    e.device = dev;
    e.n = S.n;
    e.precision = prec;
    e.wpe = shapes[best];
    char buf[1024];
    snprintf(buf, sizeof buf,
             "{\"device\": \"%s\", \"n_states\": %d, \"precision\": %d, \"waves_per_simd\": %d, "
             "\"conditions\": %d, \"shapes\": [%d, %d, %d], \"ms\": [%.3f, %.3f, %.3f]}",
             dev.c_str(), S.n, prec, shapes[best], NUM, shapes[0], shapes[1], shapes[2], ms[0], ms[1], ms[2]);
    e.line = buf;
    bool replaced = false;
    for (auto& x : entries)
      if (x.device == dev && x.n == e.n && x.precision == prec) {
        x = e;
        replaced = true;
      }
    if (!replaced) entries.push_back(e);
    if (!write_tuning(cache_path, entries)) {
      set_err("accelerInt_autotune: cannot write %s", cache_path);
      return -1;
    }
  }
  return shapes[best];
}

// Applies the cache entries of this device (any system size and precision).
// Returns the number of entries applied, or -1.
int accelerInt_load_tuning(const char* cache_path) {
  if (!ensure_init()) return -1;
  if (!cache_path) {
    set_err("accelerInt_load_tuning: no path");
    return -1;
  }
  const std::string dev = device_key();
  int applied = 0;
  for (const TuneEntry& e : read_tuning(cache_path)) {
    if (e.device != dev) continue;
    const int sys = e.n == 2 ? 0 : (e.n == 14 ? 1 : -1);
    if (sys < 0 || (e.precision != 0 && e.precision != 1)) continue;
    const int* shapes = sys == 0 ? kShapesVdp : kShapesK14;
    if (e.wpe != shapes[0] && e.wpe != shapes[1] && e.wpe != shapes[2]) continue;
    S.wpe[sys][e.precision] = e.wpe;
    ++applied;
  }
  return applied;
}

int accelerInt_set_learned_start(int on) {
  if (on) {
    const MlpView v = mlp_view();
    if (!v.on || v.n != S.n) {
      set_err("accelerInt_set_learned_start: no network for a %d-state system (accelerInt_mlp_init / _train first)", S.n);
      return -1;
    }
    if (S.n >= 64 || (S.mech == ACCELERINT_MECH_KINETICS && S.n != 54)) {
      set_err("accelerInt_set_learned_start: the learned start runs with one condition per wavefront (54-state kinetics)");
      return -1;
    }
  }
  S.learned = on ? 1 : 0;
  return 0;
}

int accelerInt_start_log(int capacity) {
  if (!ensure_init()) return -1;
  if (capacity <= 0) {
    set_err("accelerInt_start_log: capacity must be positive");
    return -1;
  }
  if (S.own_log_x) hipFree(S.own_log_x);
  if (S.own_log_z) hipFree(S.own_log_z);
  if (S.own_log_n) hipFree(S.own_log_n);
  S.own_log_x = S.own_log_z = nullptr;
  S.own_log_n = nullptr;
  if (!HIPOK(hipMalloc(&S.own_log_x, (size_t)capacity * (S.n + 2) * sizeof(float))) ||
      !HIPOK(hipMalloc(&S.own_log_z, (size_t)capacity * 3 * S.n * sizeof(float))) ||
      !HIPOK(hipMalloc(&S.own_log_n, sizeof(int))) || !HIPOK(hipMemset(S.own_log_n, 0, sizeof(int))))
    return -1;
  S.own_log_cap = capacity;
  S.P.log = StartLog{S.own_log_x, S.own_log_z, S.own_log_n, capacity};
  return 0;
}

int accelerInt_read_log(float* x_host, float* z_host, int capacity) {
  if (S.device < 0 || !S.own_log_n) {
    set_err("accelerInt_read_log: no library-owned log (accelerInt_start_log)");
    return -1;
  }
  int n = 0;
  if (!HIPOK(hipStreamSynchronize(S.stream)) || !HIPOK(hipDeviceSynchronize()) ||
      !HIPOK(hipMemcpy(&n, S.own_log_n, sizeof(int), hipMemcpyDeviceToHost)))
    return -1;
  if (n > S.own_log_cap) n = S.own_log_cap;
  if (n > capacity) n = capacity;
  if (n > 0 && ((x_host && !HIPOK(hipMemcpy(x_host, S.own_log_x, (size_t)n * (S.n + 2) * sizeof(float),
                                             hipMemcpyDeviceToHost))) ||
                (z_host && !HIPOK(hipMemcpy(z_host, S.own_log_z, (size_t)n * 3 * S.n * sizeof(float),
                                             hipMemcpyDeviceToHost)))))
    return -1;
  hipFree(S.own_log_x);
  hipFree(S.own_log_z);
  hipFree(S.own_log_n);
  S.own_log_x = S.own_log_z = nullptr;
  S.own_log_n = nullptr;
  S.own_log_cap = 0;
  S.P.log = StartLog{nullptr, nullptr, nullptr, 0};
  return n;
}

int accelerInt_log_first_steps(float* x_dev, float* z_dev, int capacity, int* count_dev) {
  if (capacity > 0 && (!x_dev || !z_dev || !count_dev)) {
    set_err("accelerInt_log_first_steps: null buffer");
    return -1;
  }
  S.P.log = capacity > 0 ? StartLog{x_dev, z_dev, count_dev, capacity} : StartLog{nullptr, nullptr, nullptr, 0};
  return 0;
}

int accelerInt_set_const_time_step(int on) {
  S.P.const_time_step = on ? 1 : 0;
  return 0;
}

int accelerInt_set_abort_on_error(int on) {
  const int prev = S.abort_on_error;
  S.abort_on_error = on ? 1 : 0;
  return prev;
}

int accelerInt_num_states(void) { return S.n; }

// solver_interface.cu:152-211
void accelerInt_initialize(int NUM, int device) {
  S.err.clear();  // void entry points report failure only through the last error
  device = device < 0 ? 0 : device;
  int num_devices = 0;
  if (hipGetDeviceCount(&num_devices) != hipSuccess) num_devices = 0;
  if (!(device >= 0 && device < num_devices)) {
    printf("Error: GPU device number not in correct range\n");
    printf("Provide number between 0 and %i\n", num_devices - 1);
    exit(1);
  }
  if (!HIPOK(hipSetDevice(device))) return;
  // the noalloc entry point's scratch array: its address on this device
  if (device < kMaxDevices && !g_noalloc_scratch[device]) {
    void* p = nullptr;
    if (!HIPOK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)))) return;
    g_noalloc_scratch[device] = static_cast<int*>(p);
  }
  if (S.mech == ACCELERINT_MECH_KINETICS) {
    std::string msg;
    for (KineticsHost* kin : {&S.kin14, &S.kin54, &S.kin112}) {
      if (kin->ns == 0) continue;
      if (!kin->upload(&msg)) {
        set_err("%s", msg.c_str());
        if (S.abort_on_error) {
          fprintf(stderr, "%s\n", msg.c_str());
          exit(-1);
        }
        return;
      }
    }
    S.kp14 = S.kin14.params<14>();
    S.kp54 = S.kin54.params<54>();
    S.kp112 = S.kin112.params<112>();
  }
  if (!HIPOK(hipStreamCreateWithFlags(&S.stream, hipStreamNonBlocking))) return;
  size_t free_mem = 0, total_mem = 0;
  if (!HIPOK(hipMemGetInfo(&free_mem, &total_mem))) return;
  const long long max_cond = (long long)floor(0.8 * (double)free_mem / (double)bytes_per_condition());
  long long cap = NUM > 0 ? NUM : 1;
  if (cap > max_cond) cap = max_cond;
  cap = ((cap + kBlock - 1) / kBlock) * kBlock;
  if (cap <= 0) {
    printf("Mechanism is too large to fit into global CUDA memory... exiting.");
    exit(-1);
  }
  S.device = device;
  if (!alloc_buffers((int)cap)) {
    S.device = -1;
    return;
  }
  S.have_status = 0;
  // launch shapes recorded by accelerInt_autotune for this device
  if (const char* cache = getenv("ACCELERINT_TUNE_CACHE")) accelerInt_load_tuning(cache);
}

// solver_interface.cu:225-275, with the batches of `padded` conditions kept and
// the transfers done as one contiguous copy plus a device transposition.
void accelerInt_integrate(const int NUM, const double t_start, const double t_end,
                          const double stepsize, double* y_host, const double* var_host) {
  S.err.clear();
  if (!ensure_init()) return;
  const int n = S.n;
  int num_solved = 0;
  if ((int)S.h_codes.size() < NUM) S.h_codes.assign(NUM, 0);
  // batches of different conditions: one batch's measured work says nothing
  // about the next one's, so batched calls take conditions in index order
  const int schedule = S.schedule;
  if (NUM > S.padded) {
    S.schedule = ACCELERINT_SCHEDULE_INDEX;
    S.cost_num = S.order_num = 0;
  }
  struct RestoreSchedule {
    int mode;
    ~RestoreSchedule() { S.schedule = mode; }
  } restore{schedule};
  std::vector<int> all_codes(NUM, 0);
  std::vector<double> stage;
  while (num_solved < NUM) {
    const int num_cond = NUM - num_solved < S.padded ? NUM - num_solved : S.padded;
    if (!HIPOK(hipMemcpyAsync(S.d_pr, var_host + num_solved, num_cond * sizeof(double),
                              hipMemcpyHostToDevice, S.stream)))
      return;
    // rows i of the caller's column-major array, columns [num_solved, +num_cond)
    if (!HIPOK(hipMemcpy2DAsync(S.d_ycm, (size_t)num_cond * sizeof(double), y_host + num_solved,
                                (size_t)NUM * sizeof(double), (size_t)num_cond * sizeof(double), n,
                                hipMemcpyHostToDevice, S.stream)))
      return;
    const size_t tot = (size_t)num_cond * n;
    const int tb = 256;
    const int nb = (int)((tot + tb - 1) / tb);
    hipLaunchKernelGGL(k_cm_to_cond, dim3(nb), dim3(tb), 0, S.stream, S.d_ycm, S.d_y, num_cond, n,
                       num_cond);
    if (!HIPOK(hipGetLastError())) return;
    if (run_steps(num_cond, t_start, t_end, stepsize, S.d_y, S.d_pr, S.d_codes,
                  S.d_cnt + (size_t)0, S.stream) != 0)
      return;
    hipLaunchKernelGGL(k_cond_to_cm, dim3(nb), dim3(tb), 0, S.stream, S.d_y, S.d_ycm, num_cond, n,
                       num_cond);
    if (!HIPOK(hipGetLastError())) return;
    if (!HIPOK(hipMemcpyAsync(all_codes.data() + num_solved, S.d_codes, num_cond * sizeof(int),
                              hipMemcpyDeviceToHost, S.stream)))
      return;
    if (!HIPOK(hipMemcpy2DAsync(y_host + num_solved, (size_t)NUM * sizeof(double), S.d_ycm,
                                (size_t)num_cond * sizeof(double), (size_t)num_cond * sizeof(double),
                                n, hipMemcpyDeviceToHost, S.stream)))
      return;
    if (!HIPOK(hipStreamSynchronize(S.stream))) return;
    num_solved += num_cond;
  }
  S.h_codes.assign(all_codes.begin(), all_codes.end());
  S.have_status = 1;
  if (S.abort_on_error) check_error(NUM, all_codes.data());
}

void intDriver(const int NUM, const double t, const double t_end, const double* pr_global,
               double* y_global) {
  if (!ensure_init()) return;
  accelerInt_integrate(NUM, t, t_end, t_end - t, y_global, pr_global);
}

int accelerInt_integrate_device_hetero3(int NUM112, double* y112_dev, const double* var112_dev, int* codes112_dev,
                                        int NUM54, double* y54_dev, const double* var54_dev, int* codes54_dev,
                                        int NUM14, double* y14_dev, const double* var14_dev, int* codes14_dev,
                                        double t_start, double t_end, double stepsize, void* stream) {
  if (!ensure_init()) return -1;
  if (S.mech != ACCELERINT_MECH_KINETICS || S.kin14.ns != 13 || S.kin54.ns != 53 ||
      (NUM112 > 0 && S.kin112.ns != 111)) {
    set_err("heterogeneous launch: install the 14- and 54-state networks (and the 112-state one for its batch) "
            "before initialize");
    return -2;
  }
  if (NUM14 < 0 || NUM54 < 0 || NUM112 < 0 || NUM14 > S.padded || NUM54 > S.padded || NUM112 > S.padded ||
      (NUM14 > 0 && (!y14_dev || !var14_dev)) || (NUM54 > 0 && (!y54_dev || !var54_dev)) ||
      (NUM112 > 0 && (!y112_dev || !var112_dev))) {
    set_err("heterogeneous launch: bad arguments (each batch at most %d conditions)", S.padded);
    return -2;
  }
  if (S.jacobian != ACCELERINT_JACOBIAN_ANALYTIC) {
    set_err("heterogeneous launch: the heterogeneous launch uses the analytic Jacobian only");
    return -2;
  }
  const double step = stepsize < 0 ? t_end - t_start : stepsize;
  if (!(t_start + kRoundoff < t_end) || NUM14 + NUM54 + NUM112 == 0) return 0;
#if !ACC_BUILTINS
  set_err("heterogeneous launch: a user-mechanism build carries one mechanism");
  return -2;
#else
  hipStream_t s = stream ? (hipStream_t)stream : S.stream;
  g_launch_msg.clear();
  // the zero Newton start, and no training-sample log: a log is sized for one
  // system and the queues' records would interleave in it
  SolverParams P = S.P;
  P.mlp = MlpView{};
  P.log = StartLog{nullptr, nullptr, nullptr, 0};
  hipError_t e = S.precision == ACCELERINT_PRECISION_MIXED
                     ? launch_hetero<float>(NUM112, var112_dev, y112_dev, codes112_dev, NUM54, var54_dev, y54_dev,
                                            codes54_dev, NUM14, var14_dev, y14_dev, codes14_dev, t_start, t_end, step,
                                            P, s)
                     : launch_hetero<double>(NUM112, var112_dev, y112_dev, codes112_dev, NUM54, var54_dev, y54_dev,
                                             codes54_dev, NUM14, var14_dev, y14_dev, codes14_dev, t_start, t_end,
                                             step, P, s);
  if (e != hipSuccess && !g_launch_msg.empty()) {
    set_err("%s", g_launch_msg.c_str());
    return -1;
  }
  return hip_ok(e, "k_radau_hetero launch") ? 0 : -1;
#endif
}

int accelerInt_integrate_device_hetero(int NUM14, double* y14_dev, const double* var14_dev, int* codes14_dev,
                                       int NUM54, double* y54_dev, const double* var54_dev, int* codes54_dev,
                                       double t_start, double t_end, double stepsize, void* stream) {
  return accelerInt_integrate_device_hetero3(0, nullptr, nullptr, nullptr, NUM54, y54_dev, var54_dev, codes54_dev,
                                             NUM14, y14_dev, var14_dev, codes14_dev, t_start, t_end, stepsize,
                                             stream);
}

int accelerInt_integrate_device(int NUM, double t_start, double t_end, double stepsize,
                                double* y_dev, const double* var_dev, int* codes_dev,
                                void* stream) {
  if (!ensure_init()) return -1;
  if (NUM < 0 || (NUM > 0 && (!y_dev || !var_dev))) {
    set_err("accelerInt_integrate_device: bad arguments");
    return -2;
  }
  hipStream_t s = stream ? (hipStream_t)stream : S.stream;
  uint32_t* cnt = (NUM <= S.padded) ? S.d_cnt : nullptr;
  return run_steps(NUM, t_start, t_end, stepsize, y_dev, var_dev, codes_dev, cnt, s);
}

int accelerInt_integrate_device_noalloc(int NUM, double t_start, double t_end, double stepsize,
                                        double* y_dev, const double* var_dev, int* codes_dev, void* stream) {
  if (S.device < 0) {
    set_err("accelerInt_integrate_device_noalloc: call accelerInt_initialize first (it installs the mechanism "
            "and locates the scratch array)");
    return -1;
  }
  if (NUM < 0 || NUM > kNoAllocMaxConditions || (NUM > 0 && (!y_dev || !var_dev))) {
    set_err("accelerInt_integrate_device_noalloc: bad arguments (NUM must be 0..%d, the scratch array's capacity)",
            kNoAllocMaxConditions);
    return -2;
  }
  int* sc = S.device < kMaxDevices ? g_noalloc_scratch[S.device] : nullptr;
  if (!sc) {
    set_err("accelerInt_integrate_device_noalloc: no scratch array on device %d", S.device);
    return -1;
  }
  const double step = stepsize < 0 ? t_end - t_start : stepsize;
  if (!(t_start + kRoundoff < t_end) || NUM == 0) return 0;
  hipStream_t s = stream ? (hipStream_t)stream : S.stream;
  const hipError_t e = launch_noalloc(NUM, t_start, t_end, step, var_dev, y_dev, codes_dev, sc, s);
  if (e != hipSuccess && !g_launch_msg.empty()) {
    set_err("%s", g_launch_msg.c_str());
    return -1;
  }
  return hip_ok(e, "k_radau launch (noalloc)") ? 0 : -1;
}

int accelerInt_eval_callbacks(int NUM, double t, const double* y_host, const double* var_host,
                              double* dy_host, double* jac_host) {
  if (!ensure_init()) return -1;
  if (NUM <= 0 || NUM > S.padded || !y_host || !var_host || !dy_host || !jac_host) {
    set_err("accelerInt_eval_callbacks: bad arguments (NUM must be 1..%d)", S.padded);
    return -2;
  }
  const int n = S.n;
  double *d_dy = nullptr, *d_jac = nullptr;
  char* d_gws = nullptr;  // the 112-state network's Jacobian workspace, one slice per condition
  if (!HIPOK(hipMalloc(&d_dy, (size_t)NUM * n * sizeof(double)))) return -1;
  if (!HIPOK(hipMalloc(&d_jac, (size_t)NUM * n * n * sizeof(double))) ||
      (n == 112 && !HIPOK(hipMalloc(&d_gws, (size_t)NUM * MechGlobal<MechKinetics112>::value * sizeof(double))))) {
    hipFree(d_dy);
    hipFree(d_jac);
    return -1;
  }
  int rc = 0;
  const size_t tot = (size_t)NUM * n;
  const int nb = (int)((tot + 255) / 256);
  std::vector<double> dy_cm((size_t)NUM * n);
  if (!HIPOK(hipMemcpyAsync(S.d_pr, var_host, NUM * sizeof(double), hipMemcpyHostToDevice, S.stream)) ||
      !HIPOK(hipMemcpyAsync(S.d_ycm, y_host, tot * sizeof(double), hipMemcpyHostToDevice, S.stream))) {
    rc = -1;
  } else {
    hipLaunchKernelGGL(k_cm_to_cond, dim3(nb), dim3(256), 0, S.stream, S.d_ycm, S.d_y, NUM, n, NUM);
    if (!hip_ok(launch_eval_any(NUM, t, S.d_pr, S.d_y, d_dy, d_jac, S.stream, d_gws), "k_eval_callbacks"))
      rc = -1;
    else {
      hipLaunchKernelGGL(k_cond_to_cm, dim3(nb), dim3(256), 0, S.stream, d_dy, S.d_ycm, NUM, n, NUM);
      if (!HIPOK(hipMemcpyAsync(dy_host, S.d_ycm, tot * sizeof(double), hipMemcpyDeviceToHost, S.stream)) ||
          !HIPOK(hipMemcpyAsync(jac_host, d_jac, tot * n * sizeof(double), hipMemcpyDeviceToHost, S.stream)) ||
          !HIPOK(hipStreamSynchronize(S.stream)))
        rc = -1;
    }
  }
  hipFree(d_dy);
  hipFree(d_jac);
  hipFree(d_gws);
  return rc;
}

int accelerInt_factor_test(int n, int precision, int NUM, const double* a_re, const double* a_im, const double* b_re,
                           const double* b_im, double* lu_re, double* lu_im, int* ipiv, int* info, double* x_re,
                           double* x_im) {
  if (!ensure_init()) return -1;
  const int max_num = n == 112 ? 4096 : (1 << 20);
  if ((n != 2 && n != 14 && n != 54 && n != 112) || NUM <= 0 || NUM > max_num || !a_re || !lu_re || !ipiv ||
      !info || (a_im && !lu_im) || (b_re && !x_re) || (a_im && b_re && (!b_im || !x_im)) ||
      (precision != ACCELERINT_PRECISION_FP64 && precision != ACCELERINT_PRECISION_MIXED)) {
    set_err("accelerInt_factor_test: bad arguments (n must be 2, 14, 54 or 112; NUM 1..%d)", max_num);
    return -2;
  }
  const bool cplx = a_im != nullptr, solve = b_re != nullptr;
  const size_t mat = (size_t)NUM * n * n, vec = (size_t)NUM * n;
  double *d_are = nullptr, *d_aim = nullptr, *d_lre = nullptr, *d_lim = nullptr;
  double *d_bre = nullptr, *d_bim = nullptr, *d_xre = nullptr, *d_xim = nullptr;
  int *d_perm = nullptr, *d_info = nullptr;
  char* d_ws = nullptr;
  int rc = 0;
  std::vector<int> perm(vec);
  const size_t ws_bytes = factor_test_ws_bytes(n) * (size_t)NUM;
  if (!HIPOK(hipMalloc(&d_are, mat * sizeof(double))) || !HIPOK(hipMalloc(&d_lre, mat * sizeof(double))) ||
      (cplx && (!HIPOK(hipMalloc(&d_aim, mat * sizeof(double))) || !HIPOK(hipMalloc(&d_lim, mat * sizeof(double))))) ||
      (solve && (!HIPOK(hipMalloc(&d_bre, vec * sizeof(double))) || !HIPOK(hipMalloc(&d_xre, vec * sizeof(double))))) ||
      (solve && cplx &&
       (!HIPOK(hipMalloc(&d_bim, vec * sizeof(double))) || !HIPOK(hipMalloc(&d_xim, vec * sizeof(double))))) ||
      !HIPOK(hipMalloc(&d_perm, vec * sizeof(int))) || !HIPOK(hipMalloc(&d_info, NUM * sizeof(int))) ||
      (ws_bytes && !HIPOK(hipMalloc(&d_ws, ws_bytes)))) {
    rc = -1;
  } else if (!HIPOK(hipMemcpyAsync(d_are, a_re, mat * sizeof(double), hipMemcpyHostToDevice, S.stream)) ||
             (cplx && !HIPOK(hipMemcpyAsync(d_aim, a_im, mat * sizeof(double), hipMemcpyHostToDevice, S.stream))) ||
             (solve && !HIPOK(hipMemcpyAsync(d_bre, b_re, vec * sizeof(double), hipMemcpyHostToDevice, S.stream))) ||
             (solve && cplx &&
              !HIPOK(hipMemcpyAsync(d_bim, b_im, vec * sizeof(double), hipMemcpyHostToDevice, S.stream)))) {
    rc = -1;
  } else if (!hip_ok(launch_factor_test(n, precision == ACCELERINT_PRECISION_MIXED, cplx, NUM, d_are, d_aim, d_bre,
                                        d_bim, d_lre, d_lim, d_perm, d_info, d_xre, d_xim, d_ws, S.stream),
                     "k_factor_test")) {
    rc = -1;
  } else if (!HIPOK(hipMemcpyAsync(lu_re, d_lre, mat * sizeof(double), hipMemcpyDeviceToHost, S.stream)) ||
             (cplx && !HIPOK(hipMemcpyAsync(lu_im, d_lim, mat * sizeof(double), hipMemcpyDeviceToHost, S.stream))) ||
             (solve && !HIPOK(hipMemcpyAsync(x_re, d_xre, vec * sizeof(double), hipMemcpyDeviceToHost, S.stream))) ||
             (solve && cplx &&
              !HIPOK(hipMemcpyAsync(x_im, d_xim, vec * sizeof(double), hipMemcpyDeviceToHost, S.stream))) ||
             !HIPOK(hipMemcpyAsync(perm.data(), d_perm, perm.size() * sizeof(int), hipMemcpyDeviceToHost, S.stream)) ||
             !HIPOK(hipMemcpyAsync(info, d_info, NUM * sizeof(int), hipMemcpyDeviceToHost, S.stream)) ||
             !HIPOK(hipStreamSynchronize(S.stream))) {
    rc = -1;
  } else {
    // pivot rows -> LAPACK interchanges: at[p] = original row now at position
    // p, where[r] = position of original row r; step k swaps positions k and
    // where[perm[k]]
    std::vector<int> at(n), where(n);
    for (int c = 0; c < NUM && rc == 0; ++c) {
      for (int i = 0; i < n; ++i) at[i] = where[i] = i;
      for (int k = 0; k < n; ++k) {
        const int r = perm[(size_t)c * n + k];
        if (r < 0 || r >= n || where[r] < k) {
          set_err("accelerInt_factor_test: matrix %d: pivot row %d at step %d is not a remaining row", c, r, k);
          rc = -3;
          break;
        }
        const int p = where[r], sw = at[k];
        ipiv[(size_t)c * n + k] = p + 1;
        at[p] = sw;
        where[sw] = p;
        at[k] = r;
        where[r] = k;
      }
    }
  }
  hipFree(d_are);
  hipFree(d_aim);
  hipFree(d_lre);
  hipFree(d_lim);
  hipFree(d_bre);
  hipFree(d_bim);
  hipFree(d_xre);
  hipFree(d_xim);
  hipFree(d_perm);
  hipFree(d_info);
  hipFree(d_ws);
  return rc;
}

int accelerInt_escalated(void) {
  if (S.device < 0 || !S.d_esc) return -1;
  int n = 0;
  if (!HIPOK(hipStreamSynchronize(S.stream))) return -1;
  if (!HIPOK(hipMemcpy(&n, S.d_esc, sizeof(int), hipMemcpyDeviceToHost))) return -1;
  return n;
}

// hipGraph of one device-resident integration (all of its kernel launches:
// work-counter resets, the persistent kernel, the FP64 escalation pass).  For
// autonomous right-hand sides such as the kinetics networks, each replay
// advances the states by the captured interval, so repeated global steps run
// as graph launches with no per-step host work.
int accelerInt_graph_capture(int NUM, double t_start, double t_end, double stepsize, double* y_dev,
                             const double* var_dev, int* codes_dev, void* stream) {
  if (!ensure_init()) return -1;
  if (NUM <= 0 || NUM > S.padded || !y_dev || !var_dev) {
    set_err("accelerInt_graph_capture: bad arguments (NUM must be 1..%d)", S.padded);
    return -2;
  }
  if (S.P.log.cap > 0) {
    // the graph would keep writing into the log's buffers after they are read and freed
    set_err("accelerInt_graph_capture: not while a training-sample log is active");
    return -2;
  }
  accelerInt_graph_release();
  hipStream_t s = stream ? (hipStream_t)stream : S.stream;
  // the occupancy queries and the queue sort run outside the capture; the
  // graph keeps its own copy of the order
  if (!hip_ok(launch(0, t_start, t_end, stepsize, var_dev, y_dev, codes_dev, nullptr, s), "occupancy query"))
    return -1;
  if (const int* order = queue_order(NUM, s)) {
    if (!HIPOK(hipMalloc(&S.graph_order, (size_t)NUM * sizeof(int))) ||
        !HIPOK(hipMemcpyAsync(S.graph_order, order, (size_t)NUM * sizeof(int), hipMemcpyDeviceToDevice, s))) {
      accelerInt_graph_release();
      return -1;
    }
    S.graph_order_num = NUM;
  }
  S.graph_mlp_gen = S.learned ? mlp_generation() : -1;
  if (!HIPOK(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed))) return -1;
  S.capturing = true;
  const int rc = run_steps(NUM, t_start, t_end, stepsize, y_dev, var_dev, codes_dev, nullptr, s);
  S.capturing = false;
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(s, &g);
  if (rc != 0 || !HIPOK(e)) {
    if (g) hipGraphDestroy(g);
    accelerInt_graph_release();
    return -1;
  }
  S.graph = g;
  if (!HIPOK(hipGraphInstantiate(&S.graph_exec, S.graph, nullptr, nullptr, 0))) {
    hipGraphDestroy(S.graph);
    S.graph = nullptr;
    S.graph_exec = nullptr;
    return -1;
  }
  return 0;
}

int accelerInt_graph_launch(int repeats, void* stream) {
  if (!S.graph_exec || repeats < 0) {
    set_err("accelerInt_graph_launch: no captured graph");
    return -1;
  }
  if (S.graph_mlp_gen >= 0 && S.graph_mlp_gen != mlp_generation()) {
    // the captured launch reads the start network's buffers, which were freed since
    set_err("accelerInt_graph_launch: the start network was re-initialized or released since capture");
    return -1;
  }
  hipStream_t s = stream ? (hipStream_t)stream : S.stream;
  for (int r = 0; r < repeats; ++r)
    if (!HIPOK(hipGraphLaunch(S.graph_exec, s))) return -1;
  return 0;
}

int accelerInt_graph_release(void) {
  if (S.graph_exec) hipGraphExecDestroy(S.graph_exec);
  if (S.graph) hipGraphDestroy(S.graph);
  if (S.graph_order) hipFree(S.graph_order);
  S.graph_exec = nullptr;
  S.graph = nullptr;
  S.graph_order = nullptr;
  S.graph_order_num = 0;
  S.graph_mlp_gen = -1;
  return 0;
}

int accelerInt_synchronize(void) {
  if (S.device < 0) return 0;
  return HIPOK(hipStreamSynchronize(S.stream)) ? 0 : -1;
}

void accelerInt_cleanup(void) {
  S.err.clear();
  if (S.device < 0) return;
  hipStreamSynchronize(S.stream);
  accelerInt_graph_release();
  free_buffers();
  S.kin14.release();
  S.kin54.release();
  S.kin112.release();
  hipStreamDestroy(S.stream);
  S.stream = nullptr;
  S.device = -1;
  S.have_status = 0;
}

int accelerInt_get_status(int* codes, int num) {
  if (!S.have_status) return -1;
  int bad = 0;
  const int m = num < (int)S.h_codes.size() ? num : (int)S.h_codes.size();
  for (int i = 0; i < m; ++i) {
    if (codes) codes[i] = S.h_codes[i];
    if (S.h_codes[i] != 0) ++bad;
  }
  return bad;
}

int accelerInt_get_counters(uint32_t* out, int num) {
  if (S.device < 0 || num > S.padded) return -1;
  if (!HIPOK(hipStreamSynchronize(S.stream))) return -1;
  return HIPOK(hipMemcpy(out, S.d_cnt, (size_t)num * NCNT * sizeof(uint32_t), hipMemcpyDeviceToHost))
             ? 0
             : -1;
}

int accelerInt_reset_counters(void) {
  if (S.device < 0) return -1;
  return HIPOK(hipMemsetAsync(S.d_cnt, 0, (size_t)S.padded * NCNT * sizeof(uint32_t), S.stream))
             ? 0
             : -1;
}

const char* accelerInt_last_error(void) { return S.err.c_str(); }

// radau2a_init.cu:28-31
const char* solver_name(void) { return "radau2a-int-gpu"; }

size_t required_solver_size(void) {
  // condition-major state + staging + return code + counters; the Radau
  // workspace itself (E1, E2, stages, interpolant) is register/LDS resident.
  return (size_t)S.n * sizeof(double) * 2 + sizeof(int) + NCNT * sizeof(uint32_t);
}

// The mechanism's per-condition device memory.  Built-in mechanisms: the
// parameter (their tables are shared by all conditions, their callback
// buffers are on chip).  A user mechanism: what examples/van_der_pol/
// gpu_memory.cu:17-29 counts -- y, dy, the parameter and the Jacobian of the
// condition being evaluated -- which here sit in the lane group's LDS slice
// (registers for up to 4 states) while the condition is integrated.
size_t required_mechanism_size(void) {
#if ACC_BUILTINS
  return sizeof(double);
#else
  return ((size_t)2 * kUserN + 1 + (size_t)kUserN * kUserN) * sizeof(double);
#endif
}

// Solver hooks of the GPU flavour, generic/solver_init.cuh:24-25
// (radau2a_init.cu:83-120).  The reference allocates each condition's Radau
// workspace in global memory there; this library keeps that workspace on chip,
// so a solver_memory describes the library's own per-condition device buffers
// (state, parameter, codes, counters).  initialize_solver makes sure the
// library is initialized (on the current device) with room for `padded`
// conditions and fills a host descriptor and its device copy; cleanup_solver
// frees the two descriptors.
struct solver_memory {
  int padded;
  int n_states;
  double* y;
  double* pr;
  int* codes;
  uint32_t* counters;
};

void initialize_solver(const int padded, solver_memory** h_mem, solver_memory** d_mem) {
  if (!h_mem || !d_mem) {
    set_err("initialize_solver: null descriptor pointers");
    return;
  }
  *h_mem = nullptr;
  *d_mem = nullptr;
  if (S.device < 0 || S.padded < padded) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    if (S.device >= 0) accelerInt_cleanup();
    accelerInt_initialize(padded, dev);
    if (S.device < 0) return;
  }
  solver_memory* h = (solver_memory*)malloc(sizeof(solver_memory));
  if (!h) {
    set_err("initialize_solver: out of host memory");
    return;
  }
  *h = solver_memory{S.padded, S.n, S.d_y, S.d_pr, S.d_codes, S.d_cnt};
  solver_memory* d = nullptr;
  if (!HIPOK(hipMalloc(&d, sizeof(solver_memory))) ||
      !HIPOK(hipMemcpy(d, h, sizeof(solver_memory), hipMemcpyHostToDevice))) {
    if (d) hipFree(d);
    free(h);
    return;
  }
  *h_mem = h;
  *d_mem = d;
}

void cleanup_solver(solver_memory** h_mem, solver_memory** d_mem) {
  if (h_mem && *h_mem) {
    free(*h_mem);
    *h_mem = nullptr;
  }
  if (d_mem && *d_mem) {
    hipFree(*d_mem);
    *d_mem = nullptr;
  }
}

// The GPU-flavour entry points under names the CPU-flavour library
// (libaccelerint_cpu.so: accelerInt_initialize(int num_threads),
// accelerInt_cleanup(int num_threads), generic/solver_interface.h:29,51) can
// call without colliding with its own.
void accelerInt_gpu_initialize(int NUM, int device) { accelerInt_initialize(NUM, device); }
void accelerInt_gpu_integrate(int NUM, double t_start, double t_end, double stepsize, double* y_host,
                              const double* var_host) {
  accelerInt_integrate(NUM, t_start, t_end, stepsize, y_host, var_host);
}
void accelerInt_gpu_cleanup(void) { accelerInt_cleanup(); }
int accelerInt_gpu_capacity(void) { return S.device >= 0 ? S.padded : 0; }

void init_solver_log(void) {}
void solver_log(void) {}

// radau2a_props.cu:15-40
void check_error(int num_cond, int* codes) {
  for (int tid = 0; tid < num_cond; ++tid) {
    const int code = codes[tid];
    switch (code) {
      case EC_consecutive_steps:
        printf("During integration of ODE# %d, an error occured on too many consecutive integration steps,"
               "exiting...\n", tid);
        exit(code);
      case EC_max_steps_exceeded:
        printf("During integration of ODE# %d, the allowed number of integration steps was exceeded,"
               "exiting...\n", tid);
        exit(code);
      case EC_h_plus_t_equals_h:
        printf("During integration of ODE# %d, the stepsize 'h' was decreased such that h = t + h,"
               "exiting...\n", tid);
        exit(code);
      case EC_newton_max_iterations_exceeded:
        printf("During integration of ODE# %d, the allowed number of newton iteration steps was exceeded,"
               "exiting...\n", tid);
        exit(code);
    }
  }
}

}  // extern "C"
