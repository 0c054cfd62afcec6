/*
 * pnfam_gpu -- C ABI of the MI355X (gfx950) pnFAM iteration engine.
 *
 * One context holds the omega-independent inputs of a pnFAM solve resident in
 * HBM (HFB basis tables, Bogoliubov matrices, couplings on the quadrature
 * grid, the operator in the qp basis) and solves batches of complex
 * frequencies.  All arrays cross the boundary as host pointers in the
 * reference's storage conventions:
 *   - state-major tables (nghl x dqp), column-major, as hfbtho_solution.f90:88-98;
 *   - block matrices as pnfam_type_blockmatrix.f90:19-26: one non-zero block per
 *     block row, blocks stored in increasing block-row order, column-major inside;
 *     maps are 0-based, -1 meaning "no block" (the Fortran side adds/subtracts 1).
 * Every entry point returns 0 on success and a negative PNFAM_GPU_E* code on
 * failure; pnfam_gpu_last_error() gives the message.  Entry points are not
 * re-entrant on one context; distinct contexts may be used from distinct
 * threads.
 */
#ifndef PNFAM_GPU_H
#define PNFAM_GPU_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PNFAM_GPU_OK 0
#define PNFAM_GPU_EINVAL -1   /* bad argument or inconsistent block structure */
#define PNFAM_GPU_EDEVICE -2  /* HIP runtime / device failure */
#define PNFAM_GPU_ESTATE -3   /* call out of order (e.g. solve before set_operator) */
#define PNFAM_GPU_ENOMEM -4   /* device allocation failed */

typedef struct pnfam_gpu_ctx pnfam_gpu_ctx;

/* omega-independent HFB / functional inputs.  Replaces the module state the
 * reference's calc_hamiltonian reads implicitly (hfb_solution: wf tables,
 * U/V/E, num_spin_up; pnfam_interaction: couplings), pnfam_setup.f90:276-321,
 * hfbtho_solution.f90:137-395, pnfam_interaction.f90:250-257. */
typedef struct {
  int32_t nb;                 /* blocks of the doubled basis (Omega>0 then TR copies) */
  int32_t dqp;                /* sum(db) */
  int32_t nghl;               /* quadrature points */
  const int32_t *db;          /* [nb] block sizes */
  const int32_t *num_spin_up; /* [nb] spin-up states lead each block */
  const int32_t *ns;          /* [dqp] 2*spin projection (+1/-1) */
  const double *wf, *wfdr, *wfdz, *wfdp, *wfd2_all; /* [nghl x dqp] column-major */
  const double *wdcori;       /* [nghl] inverse quadrature weight x Jacobian */
  const double *Ep, *En;      /* [dqp] qp energies (0 above the pairing window) */
  const double *Up, *Vp, *Un, *Vn; /* [sum db^2]; V maps block i <-> i +- nb/2 */
  const double *crho, *cs, *cpair, *cspair; /* [nghl] density-dependent couplings */
  const double *cscal;        /* [12] cdrho ctau ctj0 ctj1 ctj2 crdj cds ct cj cgs cf csdj */
} pnfam_gpu_basis;

typedef struct {
  int32_t max_iter;           /* /solver/ max_iter (pnfam_setup.f90:98-108) */
  double convergence_epsilon; /* max-abs residual threshold (1e-7) */
  int32_t broyden_history;    /* M; <0 disables mixing */
  double quench;              /* quench_residual_int; 0 skips the residual interaction */
  double alpha_mix;           /* linear mixing factor of the Broyden step */
  int32_t precision;          /* PNFAM_GPU_FP64, PNFAM_GPU_MIXED or PNFAM_GPU_MIXED_NOREFINE */
} pnfam_gpu_opts;

/* Precision of the residual interaction (the reference computes everything in
 * FP64; pnfam_solver.f90:93-221).
 *   FP64: every step in FP64.
 *   MIXED: the hamiltonian is linear in the amplitudes, so H(v_k) is carried as
 *     an FP64 sum of H applied to the increments v_k - v_{k-1}; each increment goes
 *     through the block transforms and the grid stage on split-BF16 MFMA with
 *     FP32 accumulation.  The residual, its max-norm, Broyden, G(w) and S stay
 *     FP64.  When a point first
 *     meets the tolerance, one full FP64 evaluation replaces the accumulated H
 *     and the point iterates on until it meets the tolerance again; the Broyden
 *     pair formed across that evaluation is zeroed (environment
 *     PNFAM_GPU_MIX_DROP=0 keeps it).  A point that first meets the tolerance
 *     at max_iter, with no iteration left for its refinement, is reported as
 *     interrupted (-1).  The environment variables named here set the defaults
 *     of the options of pnfam_gpu_set_option.
 *   MIXED_NOREFINE: as MIXED without the final FP64 evaluation; S then carries
 *     the low-precision error of the first increments (about 1e-6 relative).
 *   Both mixed modes keep the Broyden history in FP32 (environment
 *   PNFAM_GPU_MIX_HIST=fp64 keeps it in FP64); the residual stays FP64.
 *   In both mixed modes a point whose increment, judged by its last residual,
 *   is below 3e-3 of its largest amplitude (environment PNFAM_GPU_MIX_TAU)
 *   goes through single BF16 products instead of the three split products:
 *   its rounding error is scaled down by the increment.  The grid stage runs as
 *   GEMMs against resident pair tables or as factored kernels whose cost is per
 *   point; by default each pass takes the factored kernels for groups of at
 *   most PNFAM_GPU_MIX_AUTO_N (6) points (environment PNFAM_GPU_MIX_GRID =
 *   tables | factored | auto; PNFAM_GPU_MIX_TRIPROD = bf16 | fp64 for the
 *   block transforms). */
#define PNFAM_GPU_FP64 0
#define PNFAM_GPU_MIXED 1
#define PNFAM_GPU_MIXED_NOREFINE 2

/* Copies the basis to the device and builds the resident tables.
 * Replaces setup_pnfam's HFB + interaction set-up (pnfam_setup.f90:134-174). */
int pnfam_gpu_create(const pnfam_gpu_basis *b, pnfam_gpu_ctx **out);

/* Sets the one-body operator f (single-particle basis, block map f_ir2c) and
 * transforms it to the qp basis, Fqp = W_p^T F W_n (beta-) or W_n^T F W_p (beta+).
 * Replaces setup_extfield + the Fqp part of init_pnfam_solver
 * (pnfam_solver.f90:556-654, 364-372).  Returns nxy through *nxy_out. */
int pnfam_gpu_set_operator(pnfam_gpu_ctx *h, int32_t beta_minus, const int32_t *f_ir2c, const double *f_elem,
                           int64_t *nxy_out);

/* Solves npts frequencies together.  Per point: strength (re_s, im_s), the
 * iteration count in the reference's convention (>=0 converged after that many
 * steps, -1 interrupted at max_iter) and the last max-abs residual.  x_out, if
 * non-null, receives the final mixed amplitudes [npts][ReX, ReY, ImX, ImY].
 * Semantics of pnfam_solver.f90:93-221 (ifam) applied to each point. */
int pnfam_gpu_solve_batch(pnfam_gpu_ctx *h, int32_t npts, const double *re_w, const double *im_w,
                          const pnfam_gpu_opts *o, double *re_s, double *im_s, int32_t *iters, double *si_final,
                          double *x_out);

/* Restart from stored amplitudes: the reference's .bin restart
 * (pnfam_solver.f90:63-71 reading qrpa_broin, si and the strength through
 * pnfam_storage.f90:300-360).  x_in [npts][ReX, ReY, ImX, ImY] are the stored
 * mixed amplitudes, si_in (may be null: 1) the stored residual, re_s_in /
 * im_s_in (may be null: 0) the stored strength.  As in ifam, a point whose
 * stored residual is below the tolerance returns at iteration 0 with the stored
 * strength; the others iterate from x_in with an empty Broyden history, and
 * their first hamiltonian is evaluated from x_in. */
int pnfam_gpu_solve_batch_restart(pnfam_gpu_ctx *h, int32_t npts, const double *re_w, const double *im_w,
                                  const pnfam_gpu_opts *o, const double *x_in, const double *si_in,
                                  const double *re_s_in, const double *im_s_in, double *re_s, double *im_s,
                                  int32_t *iters, double *si_final, double *x_out);

/* Checkpoint of the full iteration state of the last batch (solve_batch,
 * solve_batch_restart or solve_resume): amplitudes, Broyden history and Gram
 * rows, accumulated fields of the mixed path, and per point its residual,
 * strength and status.  pnfam_gpu_solve_resume continues the batch from it,
 * bitwise as if it had not been interrupted, with max_iter raised (interrupted
 * points run on, converged ones keep their result; every other option, the
 * operator and the cross-terms must be those of the checkpointed batch).  No
 * counterpart in the reference, whose restart (above) drops the history.  Any
 * other call on the context between a batch and its checkpoint_save discards
 * the state. */
int pnfam_gpu_checkpoint_size(pnfam_gpu_ctx *h, int64_t *bytes);
int pnfam_gpu_checkpoint_save(pnfam_gpu_ctx *h, void *buf, int64_t bytes);
int pnfam_gpu_solve_resume(pnfam_gpu_ctx *h, const void *buf, int64_t bytes, const pnfam_gpu_opts *o, double *re_s,
                           double *im_s, int32_t *iters, double *si_final, double *x_out);

/* Cross-term operators G_x (pnfam_solver.f90:190-203, contracted with
 * contract_bbm, pnfam_type_bbm.f90:393-421): n single-particle operators with
 * the block structure of f (g_elem [n][nxy], as f_elem), transformed to the qp
 * basis like f.  Every later batch contracts each with its points' amplitudes
 * after every iteration, S_x = -(1/pi) Tr(G_x dR); pnfam_gpu_get_crossterms
 * returns the values of the last batch, [npts][n].  n = 0 removes them. */
int pnfam_gpu_set_crossterms(pnfam_gpu_ctx *h, int32_t n, const double *g_elem);
int pnfam_gpu_get_crossterms(pnfam_gpu_ctx *h, int32_t npts, double *re_x, double *im_x);

/* ---- per-unit entry points (one frequency's arrays, host in/out) -------- */

/* One modified-Broyden step, qrpa_broyden / broyden_method
 * (pnfam_broyden.f90:96-216), on the context's device history: vout (in: the
 * new amplitudes; out: vout - vin), vin (in: the last mixed amplitudes; out:
 * the mixed update), si = max|vout - vin|, flag 'N' (no mixing, M < 0), 'L'
 * (linear, M = 0 or iter = 0) or 'B' (Broyden).  Vectors [ReX, ReY, ImX, ImY],
 * 4 nxy long; o supplies broyden_history and alpha_mix, both fixed for one
 * history (the reference passes the same ones every iteration; a change with
 * iter > 0 gives PNFAM_GPU_ESTATE).  iter = 0 starts a new history; any batch
 * or other per-unit call between steps discards it (PNFAM_GPU_ESTATE on the
 * next step with iter > 0). */
int pnfam_gpu_broyden_step(pnfam_gpu_ctx *h, const pnfam_gpu_opts *o, int32_t iter, double *vout, double *vin,
                           double *si, char *flag);


/* Block structure of the four quadrants of drho_sp and of X/Y (0-based maps):
 * maps[0..3][nb] = m11 (rho_pn), m12 (kappa+), m21 (kappa-), m22 (rho_np);
 * xy_maps[0..1][nb] = X (F20 layout), Y (F02 layout). */
int pnfam_gpu_structures(pnfam_gpu_ctx *h, int32_t *maps, int32_t *xy_maps);

/* Fqp = W^T f W for the operator set by pnfam_gpu_set_operator. */
int pnfam_gpu_get_fqp(pnfam_gpu_ctx *h, double *f20, double *f02);

/* qp -> sp transform of the amplitudes: drho_sp = W_p dR_qp W_n^T
 * (pnfam_solver.f90:144-150).  rsp: [8][nxy] re m11, im m11, re m12, ... im m22. */
int pnfam_gpu_qp2sp(pnfam_gpu_ctx *h, const double *x_re, const double *x_im, const double *y_re,
                    const double *y_im, double *rsp);

/* The 16-array calc_hamiltonian with the semantics of calc_dHsp_interface
 * (pnfam_setup.f90:56-71, pnfam_hamiltonian_blas.f90:51-74): in [8][nxy] =
 * re/im rho_pn, kappa+, rho_np, kappa- in the maps of pnfam_gpu_structures;
 * out [8][nxy] = re/im h_pn, Delta+, h_np, Delta- in the maps f, X, f, Y. */
int pnfam_gpu_calc_hamiltonian(pnfam_gpu_ctx *h, const double *in, double *out);

/* sp -> qp transform: dH_qp = W_p^T dH_sp W_n (pnfam_solver.f90:160-166);
 * hsp as the out array of pnfam_gpu_calc_hamiltonian. */
int pnfam_gpu_sp2qp(pnfam_gpu_ctx *h, const double *hsp, double *h20_re, double *h20_im, double *h02_re,
                    double *h02_im);

/* Selects the arithmetic of the per-unit entry points: PNFAM_GPU_FP64
 * (default) or PNFAM_GPU_MIXED, the split-BF16 kernels that the mixed solve
 * applies to its increments (grid stage of pnfam_gpu_calc_hamiltonian and
 * pnfam_gpu_densities in the form PNFAM_GPU_MIX_GRID selects, block transforms
 * of pnfam_gpu_qp2sp and pnfam_gpu_sp2qp).  No counterpart in the reference: a
 * parity hook for the mixed path. */
int pnfam_gpu_set_unit_precision(pnfam_gpu_ctx *h, int32_t precision);

/* Coordinate-space densities of one sector (diagnostic): dens [56][nghl],
 * 28 complex local densities (re, im interleaved by density) after the
 * quadrature weights are stripped (pnfam_hamiltonian_blas.f90:679-709). */
int pnfam_gpu_densities(pnfam_gpu_ctx *h, const double *in, int32_t sector, double *dens);

/* calc_hamiltonian for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).  No
 * counterpart in the reference.  As pnfam_gpu_calc_hamiltonian in FP64, with
 * device pointers d_in / d_out ([8][nxy] each, calc_dHsp_interface's argument
 * order); the call allocates nothing: the local densities, fields and dH_sp
 * quadrants live in the library's file-scope device scratch array of 32 MiB per
 * device (held until the process ends), and a problem needing more
 * (2 * 2 * 132 * nghl + 8 * nxy doubles) is refused with PNFAM_GPU_EINVAL.
 * Call it on the device the context was created on; it returns after the work
 * on the context's stream has finished.  Calls on one device share its scratch
 * array, so calls that overlap on one device race. */
int pnfam_gpu_calc_hamiltonian_noalloc(pnfam_gpu_ctx *h, const double *d_in, double *d_out);

/* ---- options and measurement (no counterpart in the reference) ---------- */

/* Context options, by name:
 *   unit_replicas  1..256: the per-unit entry points run their frequency in
 *                  that many batch slots (identical inputs) and return the last,
 *                  so that they take the launch paths of batches that size;
 *                  giving it (1 too) also sets unit_general;
 *   unit_general   1: the FP64 grid stage of the per-unit calls runs the
 *                  general kernels, whose launch-shape options (proj_*,
 *                  fp64_density) unit_replicas serves to compare; 0 (default
 *                  until unit_replicas is given): the form the solves take
 *                  (fp64_grid);
 *   fp64_grid      0 (default): on a basis whose wavefunction tables are
 *                  products of a radial and an axial function (found from the
 *                  tables when the context is created; the harmonic-oscillator
 *                  bases all are) the FP64 grid stage contracts one direction
 *                  at a time, in all solves and per-unit calls but
 *                  calc_hamiltonian_noalloc; 1: always the general kernels,
 *                  which contract over all grid points (results differ in
 *                  summation order; read back fp64_separable: 1 where the
 *                  first form is in use -- in per-unit calls only while
 *                  unit_general is 0 -- and 0 also after a call that took the
 *                  other one for want of memory; fp64_residual: largest
 *                  deviation of the tables from products, relative to each
 *                  table's largest value, at most 1e-14 for the first form);
 *   fp64_grid_bytes  bytes of the first form's intermediates: a batch that
 *                  needs more runs in passes of as many points as fit, and
 *                  where not one fits, or the memory cannot be had, the
 *                  general kernels run; 0 (default): 4 GiB, at least one point
 *                  a pass (read back fp64_point_bytes, the bytes of a point,
 *                  and fp64_held_bytes, what the context holds for the stage);
 *   mix_tau        one-product threshold of the mixed path (PNFAM_GPU_MIX_TAU);
 *   mix_hist64     1: the mixed path keeps its Broyden history in FP64;
 *   mix_drop       0: keep the Broyden pair formed across a refinement;
 *   mix_auto_n     points at or below which the mixed grid stage takes the
 *                  factored kernels (PNFAM_GPU_MIX_AUTO_N);
 *   mix_grid       0 auto, 1 pair tables, 2 factored (before the first mixed
 *                  call only); auto builds the pair tables only if they take
 *                  at most mix_table_frac (default 0.5) of the free device
 *                  memory, and reads back 2 when it chose the factored kernels
 *                  (mix_table_bytes: the table size it estimated);
 *   mix_refine_at  1..1e6 (default 1): the mixed path refines a point in FP64
 *                  when its residual first drops below this multiple of the
 *                  tolerance;
 *   mix_refine_every 1..64 (default 8): the refinements run on batch
 *                  iterations that are multiples of this; a point that gets
 *                  there in between waits without iterating (its iteration
 *                  count, Broyden history and result are its own; max_iter
 *                  counts batch iterations, so a point that waited can stop
 *                  with up to this many less one fewer iterations of its own);
 *   graph          1: FP64 solves replay each iteration from the third on as
 *                  one HIP graph whose first kernel runs the exit tests on the
 *                  device and writes the active list; the host launches
 *                  without reading residuals and captures a graph with fewer
 *                  slots once an eighth of the captured points has retired
 *                  (results equal the eager loop run with few_split 0);
 *   few_split      0: the FP64 grid stage never splits its grid loops for
 *                  batches of eight points or fewer (1, default: it does;
 *                  the split changes the summation order of the densities);
 *   zero_skip      1 (default): the transforms (qp -> sp, sp -> qp) and the
 *                  projection do not zero their outputs first when their
 *                  blocks or tiles cover every element (read back zero_skips,
 *                  the sum of 1 qp -> sp, 2 sp -> qp, 4 projection); 0: they
 *                  always do (results are the same);
 *   proj_rows      1..4: 16-row tiles per wave of the FP64 projection;
 *   proj_freqs     1 or 2: frequencies per wave of the FP64 projection; 4:
 *                  four waves per workgroup share the psi operands in LDS;
 *   proj_stages    1 or 2 (default): k steps of operands the FP64 projection
 *                  loads ahead of its products;
 *   proj_freqs_rt1 0 (default: as proj_freqs), 1, 2 or 4: proj_freqs for the
 *                  mean-field tiles of one 16-row tile;
 *   fp64_density   0: one wave per 16 grid points, 1: two waves splitting
 *                  the tables and exchanging the products through LDS,
 *                  2 (default): two waves splitting the rows by spin, with
 *                  transposed products and no exchange (a basis whose block
 *                  states are not spin-sorted runs 1 instead);
 *   fac_freqs      frequencies per wave of the factored BF16 projection of
 *                  the mixed path: 1, 2, or 0 (default) two from 16 points.
 * Read-only: graph_launches, graph_captures and graph_capture_ms (host
 * milliseconds spent capturing and instantiating) of the last FP64 solve;
 * refine_waits, the iterations the points of the last batch waited for their
 * refinement groups.
 * The launch-shape options change no result beyond the order in which four of
 * the 28 densities add their two spin parts (fp64_density). */
int pnfam_gpu_set_option(pnfam_gpu_ctx *h, const char *name, double value);
int pnfam_gpu_get_option(pnfam_gpu_ctx *h, const char *name, double *value);

/* Distinct kernel classes (kernel name with its template arguments,
 * separated by ';') launched since pnfam_gpu_profile last enabled profiling; *len_out
 * receives the length including the terminating zero. */
int pnfam_gpu_kernel_classes(pnfam_gpu_ctx *h, char *buf, int32_t len, int32_t *len_out);


/* Resets the per-kernel totals and turns HIP-event timing of every launch on
 * the engine stream on (enable != 0) or off. */
int pnfam_gpu_profile(pnfam_gpu_ctx *h, int32_t enable);

/* Per kernel: name (32 bytes each), total milliseconds, launches, processed
 * frequency-units (sum of active frequencies over launches) and the
 * algorithmic FLOP per frequency-unit of that kernel (0 for data movement). */
int pnfam_gpu_profile_read(pnfam_gpu_ctx *h, int32_t max_kernels, char *names, double *ms, int64_t *launches,
                           double *units, double *flops_per_unit, int32_t *n_out);

void pnfam_gpu_destroy(pnfam_gpu_ctx *h);
const char *pnfam_gpu_last_error(void);

/* Build description (arch, precision paths) for logs. */
const char *pnfam_gpu_version(void);

#ifdef __cplusplus
}
#endif
#endif
