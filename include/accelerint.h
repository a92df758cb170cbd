/*
 * accelerInt-compatible C ABI of the MI355X (gfx950) batched Radau IIA-5
 * library, libaccelerint_hip.so.
 *
 * The first group of entry points has exactly the signatures of the
 * reference's GPU library interface and solver hooks, so a caller written
 * against SLACKHA/accelerInt's radau2a GPU build links against this library
 * unchanged.  The second group is additive (no reference counterpart):
 * runtime mechanism and tolerance selection, non-aborting status reporting,
 * and a device-resident entry point whose buffers already live in HBM.
 *
 * Data layout at the boundary is the reference's: y_host is column-major,
 * y_host[i * NUM + tid] holds state component i of condition tid
 * (examples/main.dox:70-82, generic/solver_generic.c:41-44), and
 * var_host[tid] is the per-condition parameter (mu for van der Pol, pressure
 * in Pa for the kinetics networks).  y_host is updated in place.
 */
#ifndef ACCELERINT_H
#define ACCELERINT_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- reference interface ---------------------------------------------------- */

/* Replaces generic/solver_interface.cuh:35 accelerInt_initialize(int NUM, int device).
 * device < 0 selects device 0; an out-of-range device prints the reference's
 * message and exits with status 1 (solver_interface.cu:97-107). */
void accelerInt_initialize(int NUM, int device);

/* Replaces generic/solver_interface.cuh:49-50.  Integrates NUM conditions from
 * t_start to t_end in global steps of `stepsize` (stepsize < 0: one step of
 * t_end - t_start).  Global step k ends at t_start + (k+1)*stepsize, clipped to
 * t_end; the reference's own loop ignores t_start there
 * (solver_interface.cu:209), which this library does not reproduce. */
void accelerInt_integrate(const int NUM, const double t_start, const double t_end,
                          const double stepsize, double *y_host, const double *var_host);

/* Replaces generic/solver_interface.cuh:55 accelerInt_cleanup(). */
void accelerInt_cleanup(void);

/* Replaces the CPU driver generic/solver.h:32-33 intDriver(NUM, t, t_end, pr, y):
 * one global step [t, t_end] of all NUM conditions, run on the GPU, same
 * column-major y_global layout.  Initializes device 0 on first use. */
void intDriver(const int NUM, const double t, const double t_end, const double *pr_global,
               double *y_global);

/* Solver hooks, generic/solver_init.cuh:21-26 and solver_props.cuh:25-26. */
const char *solver_name(void);            /* "radau2a-int-gpu" (radau2a_init.cu:28-31) */
size_t required_solver_size(void);        /* device bytes per condition, solver part */
size_t required_mechanism_size(void);     /* device bytes per condition, mechanism part
                                             (examples/van_der_pol/gpu_memory.cu:17-29) */
void init_solver_log(void);
void solver_log(void);
/* radau2a_props.cu:15-40: prints the reference's message for the first
 * condition with a non-zero code and exits with that code. */
void check_error(int num_conditions, int *code_arr);
/* Replaces generic/solver_init.cuh:24-25 (radau2a_init.cu:83-120).  The Radau
 * workspace is on chip here, so a solver_memory describes the library's own
 * per-condition device buffers; initialize_solver initializes the library on
 * the current device with room for `padded` conditions if it is not already,
 * and returns a host descriptor and its device copy; cleanup_solver frees the
 * two descriptors (not the library). */
typedef struct solver_memory solver_memory;
void initialize_solver(const int padded, solver_memory **h_mem, solver_memory **d_mem);
void cleanup_solver(solver_memory **h_mem, solver_memory **d_mem);

/* ---- additive interface (no reference counterpart) ------------------------ */

/* Mechanism selection; must precede accelerInt_initialize.  The reference
 * compiles exactly one mechanism into each build (examples/van_der_pol/header.h:26,
 * mechanism/ for pyJac output); this library carries the van der Pol example
 * and the synthetic constant-pressure kinetics family, chosen at run time. */
#define ACCELERINT_MECH_VAN_DER_POL 0
#define ACCELERINT_MECH_KINETICS 2
/* A user mechanism's device callbacks (include/accelerint_mechanism.h),
 * compiled into a library of its own by
 *   python -m accelerint_amd.build --mechanism DIR
 * which carries that one mechanism (the default of that build) and neither
 * the van der Pol example nor the kinetics networks. */
#define ACCELERINT_MECH_USER 3
int accelerInt_select_mechanism(int kind);

/* Synthetic kinetics network (state (T, Y_1..Y_ns), N = ns + 1).  Arrays are
 * copied.  slots[6*j + 0..2] = reactant species (-1 = empty), slots[6*j + 3..5]
 * = product species; thermo[5*s + 0..4] = a0, a1, a2, bh, bs with
 * cp/R = a0 + a1 T + a2 T^2, h/R = a0 T + a1 T^2/2 + a2 T^3/3 + bh,
 * s/R = a0 ln T + a1 T + a2 T^2/2 + bs; rate constants
 * kf = exp(lnA + beta ln(T/1000) - EaR/T) in mol-cm-s units.
 * One network per compiled size (14, 54, 112) is kept (installing several
 * enables the heterogeneous launches); the most recently installed one is the
 * mechanism the other calls integrate.  The 112-state network runs one
 * condition per wavefront with its factorizations in a global workspace that
 * accelerInt_initialize allocates (blocked LU, MFMA trailing updates).
 * Returns 0, or -1 if ns + 1 is not a compiled system size. */
int accelerInt_set_kinetics(int ns, int nr, const double *W, const double *thermo,
                            const int *slots, const double *lnA, const double *beta,
                            const double *EaR);

/* ---- files of the reference's command-line driver -------------------------
 * Initial conditions (generic/read_initial_conditions.c:30-78, CONP): NUM
 * records of N + 2 doubles [t, y_0, param, y_1 .. y_{N-1}], N =
 * accelerInt_num_states() of the selected mechanism; y_host column-major
 * (y_host[i*NUM + c]), var_host[c] = param.  The reference's signature
 * allocates and exits on error; the accelerInt_ variant fills caller arrays and
 * returns 0 or -1 (message: accelerInt_last_error). */
void read_initial_conditions(const char *filename, int NUM, double **y_host, double **variable_host);
int accelerInt_read_initial_conditions(const char *filename, int NUM, double *y_host, double *var_host);
/* State log (generic/solver_main.c:47-66): t, then N doubles per condition;
 * appends unless append == 0.  Returns 0 or -1. */
int accelerInt_write_log(const char *path, int append, int NUM, double t, const double *y_host);
/* accelerInt_set_kinetics from a binary network file: int32 ns, int32 nr,
 * W[ns], thermo[ns][5], slots int32[nr][6], lnA[nr], beta[nr], EaR[nr].
 * Returns 0 or -1. */
int accelerInt_load_kinetics(const char *path);

/* Runtime tolerances (the reference's ATOL/RTOL macros; defaults 1e-10, 1e-6)
 * and the CONST_TIME_STEP switch. */
int accelerInt_set_tolerances(double atol, double rtol);
int accelerInt_set_const_time_step(int on);

/* Arithmetic of the iteration matrices.  FP64 (default): everything in double,
 * as the reference.  MIXED: the real and complex LU factorizations and the
 * Newton solves in float; dydt residuals, the error estimate (its solve gets one
 * FP64 iterative-refinement step), step control and the state stay double.
 * May be changed between integrate calls.  Returns 0, or -1 for an unknown mode. */
#define ACCELERINT_PRECISION_FP64 0
#define ACCELERINT_PRECISION_MIXED 1
int accelerInt_set_precision(int mode);

/* Jacobian of the iteration matrices: the mechanism's analytic eval_jacob
 * (default) or the reference's finite-difference one, generic/fd_jacob.c:24-127
 * (FD_ORD 1: one forward difference per column, increment
 * max(sqrt(eps)|y_j|, r0 / (atol + rtol|y_j|)) with r0 = 1000 rtol eps N
 * sqrt(sum((atol + rtol|y_i|) f_i)^2 / N)), for callbacks without an analytic
 * Jacobian.  Compiled for van der Pol and the 14- and 54-state networks
 * (single-network launches).  The learned start is compiled with the analytic
 * Jacobian only: an integration with both selected fails (-1, or the abort of
 * abort mode) instead of running another method.  May be changed between
 * integrate calls; returns 0 or -1. */
#define ACCELERINT_JACOBIAN_ANALYTIC 0
#define ACCELERINT_JACOBIAN_FINITE_DIFFERENCE 1
int accelerInt_set_jacobian(int mode);
/* Order of the finite-difference Jacobian, the reference's compile-time
 * FD_ORD (generic/fd_jacob.c:14,33-66): 1 (default, forward difference), or
 * 2, 4, 6 (central differences, order x N + 1 dydt calls per Jacobian).
 * Returns 0 or -1 for any other order. */
int accelerInt_set_fd_order(int order);

/* Launch shapes (no reference counterpart): the waves per SIMD the integration
 * kernel's register allocation targets.  van der Pol: 1, 2 (default) or 4; the
 * 14-state network: 1, 2 (default) or 3; the 54-state network: 1 only.
 * accelerInt_autotune times each shape of the selected system and precision on
 * NUM device-resident conditions (y_dev condition-major, left unchanged),
 * keeps the fastest and, if cache_path is given, records it there (a JSON array,
 * one entry per device, system size and precision); ms_out (may be NULL)
 * receives the three timings.  Returns the chosen waves per SIMD, or -1.
 * accelerInt_load_tuning applies a cache's entries for this device (returns
 * how many); accelerInt_initialize does so itself when the environment
 * variable ACCELERINT_TUNE_CACHE names a cache.  Results do not depend on the
 * shape. */
int accelerInt_set_launch_shape(int n_states, int precision, int waves_per_simd);
int accelerInt_get_launch_shape(int n_states, int precision);
int accelerInt_autotune(int NUM, double t_start, double t_end, double stepsize, const double *y_dev,
                        const double *var_dev, const char *cache_path, double *ms_out);
int accelerInt_load_tuning(const char *cache_path);

/* Order in which the persistent kernel takes conditions (no reference
 * counterpart; results do not depend on it).  LONGEST_FIRST (default): when
 * the previous integration covered the same number of conditions in one
 * batch, they are taken in decreasing order of the work each needed then
 * (greedy list scheduling: the costly conditions start first instead of
 * finishing last); otherwise, and with INDEX, in index order. */
#define ACCELERINT_SCHEDULE_INDEX 0
#define ACCELERINT_SCHEDULE_LONGEST_FIRST 1
int accelerInt_set_schedule(int mode);
/* The per-condition work of the last integration (units of one dydt call) and
 * the order the next one will use (may be NULL).  Returns the number of
 * conditions the order covers (0: index order), or -1 before initialize. */
int accelerInt_get_schedule(float *work, int *order, int num);

/* 1 (default): any non-zero condition code aborts the process through
 * check_error, as the reference does.  0: codes are kept and returned by
 * accelerInt_get_status; integration continues for the other conditions.
 * Returns the previous setting. */
int accelerInt_set_abort_on_error(int on);

/* The GPU-flavour initialize / integrate / cleanup under names that do not
 * collide with the CPU flavour's accelerInt_initialize(int num_threads) and
 * accelerInt_cleanup(int num_threads) (generic/solver_interface.h:29,51),
 * for the CPU-flavour library libaccelerint_cpu.so (include/accelerint_cpu.h),
 * which runs that interface on this library's GPU path.  capacity: the
 * conditions one launch holds (0 before initialize). */
void accelerInt_gpu_initialize(int NUM, int device);
void accelerInt_gpu_integrate(int NUM, double t_start, double t_end, double stepsize, double *y_host,
                              const double *var_host);
void accelerInt_gpu_cleanup(void);
int accelerInt_gpu_capacity(void);

/* Codes of the last integrate call (num entries); returns the count of
 * non-zero codes, or -1 if no call has been made. */
int accelerInt_get_status(int *codes, int num);

/* Per-condition event counters accumulated since initialize or the last
 * reset: out[c*10 + k], k = step, accept, reject, newton_fail, lu, lu_fail,
 * newton, f, jac, es; num at most the capacity given to initialize (a call
 * with more conditions runs in batches of that capacity, each adding into the
 * slots of its own first conditions).  Returns 0 on success. */
int accelerInt_get_counters(uint32_t *out, int num);
int accelerInt_reset_counters(void);

/* System size of the selected mechanism. */
int accelerInt_num_states(void);

/* Device-resident integration: y_dev is condition-major (y_dev[c*N + i]),
 * var_dev[c], codes_dev[c] (may be NULL) are device pointers in HBM; `stream`
 * is a hipStream_t (NULL = the library's stream).  Runs the same global-step
 * loop as accelerInt_integrate without host copies and returns without
 * waiting for completion.  Returns 0 or a negative error. */
int accelerInt_integrate_device(int NUM, double t_start, double t_end, double stepsize,
                                double *y_dev, const double *var_dev, int *codes_dev,
                                void *stream);

/* No counterpart in the reference: accelerInt_integrate_device for callers
 * that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  It calls no hipMalloc,
 * hipFree or allocating library routine: the persistent queue's work counter
 * and the list of conditions handed from the FP32-factor pass to the FP64
 * pass live in a static device array of the library (1 MiB per GPU, held
 * until the process ends), whose address accelerInt_initialize looks up on its
 * device.  Limit: NUM <= 262144 (returns -2 beyond it or for NUM < 0; -1
 * before accelerInt_initialize).  Same arguments, precision, mechanism and
 * learned start as accelerInt_integrate_device; conditions are queued in
 * index order and no event counters or per-condition costs are recorded.
 * Every call on one GPU shares that array and clears what must start at zero,
 * so calls that overlap on one GPU (two streams, two threads) race.
 * Asynchronous on `stream`.  Returns 0 or a negative error. */
int accelerInt_integrate_device_noalloc(int NUM, double t_start, double t_end, double stepsize,
                                        double *y_dev, const double *var_dev, int *codes_dev,
                                        void *stream);

/* Heterogeneous batch in one persistent launch (no reference counterpart):
 * conditions of the installed 14-state network (y14_dev[c*14 + i]) and of the
 * installed 54-state network (y54_dev[c*54 + i]) integrated together, long jobs
 * first; each batch at most NUM-at-initialize conditions; codes arrays may be
 * NULL.  Precision and tolerances as set; both parts use the zero Newton
 * start (the learned start is compiled into the single-network kernels only)
 * and the analytic Jacobian (returns -2 while the finite-difference one is
 * selected), and append nothing to an active training-sample log.
 * Asynchronous on `stream`.  Returns 0 or a negative error. */
int accelerInt_integrate_device_hetero(int NUM14, double *y14_dev, const double *var14_dev, int *codes14_dev,
                                       int NUM54, double *y54_dev, const double *var54_dev, int *codes54_dev,
                                       double t_start, double t_end, double stepsize, void *stream);
/* The same with a batch of the installed 112-state network as well
 * (y112_dev[c*112 + i]; NUM112 may be 0): every wavefront drains the 112-state
 * queue (one condition per wave; its factors and Jacobian in a library-owned
 * global workspace, allocated by accelerInt_initialize when that network is
 * installed), then the 54-state queue, then the 14-state one. */
int accelerInt_integrate_device_hetero3(int NUM112, double *y112_dev, const double *var112_dev, int *codes112_dev,
                                        int NUM54, double *y54_dev, const double *var54_dev, int *codes54_dev,
                                        int NUM14, double *y14_dev, const double *var14_dev, int *codes14_dev,
                                        double t_start, double t_end, double stepsize, void *stream);

/* Evaluates the mechanism callbacks on the device at each condition's state
 * without integrating (the reference's rate/Jacobian dump,
 * tests/rateOutputTest.cu:18): y_host/var_host as in accelerInt_integrate,
 * dy_host column-major like y_host, jac_host[c*N*N + i + j*N] the column-major
 * Jacobian of condition c.  NUM must not exceed the initialized capacity.
 * Returns 0 or a negative error. */
int accelerInt_eval_callbacks(int NUM, double t, const double *y_host, const double *var_host,
                              double *dy_host, double *jac_host);

/* Test hook, no counterpart in the reference's API: factors NUM matrices of
 * order n (2, 14, 54 or 112) on the device with the LU the integrator runs at
 * that order and precision (implicit interchanges with LAPACK's pivot rule: a
 * row per lane up to order 54, the workspace LU at 112; at order 54 the real
 * and the complex LU step by step together, the other one on the same matrix)
 * and returns them in the form of LAPACK dgetrf_ / zgetrf_, the calls of
 * RK_Decomp (radau2a.c:273,277):
 * a_re / a_im are NUM row-major n x n matrices (a_im NULL: real LU; else the
 * imaginary parts of a complex LU); lu_re / lu_im receive the combined unit-L
 * / U factors of P A, row-major; ipiv[c*n + k] the 1-based row interchanged
 * with row k at step k; info[c] the first exactly zero pivot (1-based) or 0.
 * With b_re (and b_im for a complex LU) set, the integrator's triangular
 * solves, the counterpart of dgetrs_ / zgetrs_ (radau2a.c:404,417), also run
 * on one right-hand side per matrix (b[c*n + i]) and x_re / x_im receive
 * A^-1 b; b_re NULL: no solve.  precision ACCELERINT_PRECISION_MIXED factors
 * and solves with the inputs rounded to FP32 in FP32, as the mixed-precision
 * integrator does.  Returns 0 or a negative error. */
int accelerInt_factor_test(int n, int precision, int NUM, const double *a_re, const double *a_im,
                           const double *b_re, const double *b_im, double *lu_re, double *lu_im, int *ipiv,
                           int *info, double *x_re, double *x_im);

/* Mixed precision: number of conditions of the last integration (its last
 * batch of at most NUM-at-initialize conditions) whose FP32-factor run ended
 * with a non-zero code or a non-finite state and were therefore integrated
 * again from their initial state with FP64 factors.  Waits for the library
 * stream.  Returns -1 before initialize. */
int accelerInt_escalated(void);

/* ---- learned Newton start (no reference counterpart) ------------------------
 * A small network (N + 2 -> 128 -> 128 -> 3N, GELU, BF16 MFMA with FP32
 * accumulation) predicts the stage values Z1..Z3 of the first step of each
 * global step from the features (1000/T, log Y_1..log Y_ns (floored at 1e-30),
 * log h, log p), replacing the reference's zero start (radau2a.c:600-603).
 * The zero start takes over when the first Newton correction from the
 * prediction is not smaller than the corrected stages, when Newton from it
 * fails, and after any rejection of that step; Radau's own error control
 * judges every step.  A condition whose predicted start was discarded once
 * gets the zero start for the rest of that integration call.  Features and
 * targets passed to the training calls are normalized by the caller
 * (x = (feature - mu) / sd, t = Z / zscale), the same mu, sd and zscale given
 * to accelerInt_mlp_set_normalization for use inside the integrator.
 * All return 0 on success, -1 on error (message: accelerInt_mlp_last_error). */
int accelerInt_mlp_init(int n_states, unsigned seed);
int accelerInt_mlp_param_count(void);
/* Parameters in order W1[in_p][128], b1[128], W2[128][128], b2[128],
 * W3[128][out_p], b3[out_p] with in_p = 16*ceil((N+2)/16), out_p = 16*ceil(3N/16). */
int accelerInt_mlp_get_params(float *out, int count);
int accelerInt_mlp_set_params(const float *in, int count);
int accelerInt_mlp_set_normalization(const float *mu, const float *sd, const float *zscale);
/* Mean squared error over a batch (B a multiple of 16) and its gradient
 * (host arrays: x[B][N+2], t[B][3N], grad[param_count]). */
int accelerInt_mlp_loss_grad(int B, const float *x, const float *t, float *grad, float *loss);
/* Batched forward pass (host arrays x[B][N+2] -> y[B][3N], normalized). */
int accelerInt_mlp_predict(int B, const float *x, float *y);
/* Adam on device-resident samples x_dev[n][N+2], t_dev[n][3N]; loss_per_epoch
 * (may be NULL) receives the mean squared error of each epoch. */
int accelerInt_mlp_train(int n, const float *x_dev, const float *t_dev, int epochs, int batch, float lr,
                         unsigned seed, float *loss_per_epoch);
/* The integrator's own inference path (one wavefront per condition) on given
 * states: y[num][54] condition-major, parameters pr[num], step size h ->
 * z[num][3*54] = (Z1, Z2, Z3) denormalized.  54-state networks only. */
int accelerInt_mlp_predict_states(int num, double h, const double *y, const double *pr, double *z);
/* accelerInt_mlp_train on host arrays (copied to the device for the call). */
int accelerInt_mlp_train_host(int n, const float *x, const float *t, int epochs, int batch, float lr,
                              unsigned seed, float *loss_per_epoch);
const char *accelerInt_mlp_last_error(void);
void accelerInt_mlp_release(void);
/* Use (1) or stop using (0) the trained network as the Newton start of each
 * global step's first step (54-state kinetics: one condition per wavefront). */
int accelerInt_set_learned_start(int on);
/* Training-data log: while capacity > 0, every integration appends one sample
 * per accepted first step of a global step: x_dev[i][N+2] = features of the
 * step start (as above: 1000/T, log Y_k, log h, log p), z_dev[i][3N] = converged (Z1, Z2, Z3), as float; *count_dev
 * (device int, zeroed by the caller) counts appended samples (it may exceed
 * capacity; samples beyond it are dropped).  capacity 0 turns logging off. */
int accelerInt_log_first_steps(float *x_dev, float *z_dev, int capacity, int *count_dev);
/* The same log in library-owned device buffers: start_log allocates room for
 * `capacity` samples and turns logging on; read_log copies up to `capacity`
 * samples to the host arrays, frees the buffers, turns logging off and returns
 * the number of samples copied (negative on error). */
int accelerInt_start_log(int capacity);
int accelerInt_read_log(float *x_host, float *z_host, int capacity);

/* hipGraph of one accelerInt_integrate_device call (no reference
 * counterpart): capture records every kernel launch of the call for these
 * buffers and interval; launch replays it `repeats` times on `stream` (NULL =
 * the library's stream).  With autonomous right-hand sides (the kinetics
 * networks) each replay advances the states by t_end - t_start, so a loop of
 * global steps becomes one host call.  NUM at most NUM-at-initialize.  One
 * graph at a time; capture replaces it, release (or cleanup) frees it.  The
 * graph keeps its own copy of the queue order present at capture; capture is
 * refused (-2) while a training-sample log is active, and a replay is refused
 * (-1) once the start network it reads has been re-initialized or released. */
int accelerInt_graph_capture(int NUM, double t_start, double t_end, double stepsize, double *y_dev,
                             const double *var_dev, int *codes_dev, void *stream);
int accelerInt_graph_launch(int repeats, void *stream);
int accelerInt_graph_release(void);

/* Blocks until the library stream is idle; returns 0 or a negative error. */
int accelerInt_synchronize(void);

/* Last error message recorded by the library ("" if none).  Cleared on entry
 * to accelerInt_initialize, accelerInt_integrate (and intDriver) and
 * accelerInt_cleanup, whose void signatures report failure only here. */
const char *accelerInt_last_error(void);

#ifdef __cplusplus
}
#endif

#endif
