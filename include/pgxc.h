/*
 * pgxc.h -- C ABI of the MI355X exchange-correlation grid integration.
 *
 * Drop-in boundary for the body of ParaGauss's calc_xcks_nl / calc_xcks
 * (modules/xc_hamiltonian.f90:1280-1580 and :812-1036).  Everything around
 * those routines stays in the Fortran SCF driver: xc_build's allocation and
 * zeroing (modules/xc_hamiltonian.f90:1038-1116), xc_sndrcv (:769-798),
 * xc_pseudo2d_sym, mixing and the checkpoint records.  The Fortran side binds
 * these entry points with ISO_C_BINDING (paragauss-gpl_amd/fortran/pgxc_binding.f90).
 *
 * All arrays are plain host pointers in the reference's Fortran layouts
 * (column-major, 0-based here).  Every entry point returns PGXC_OK (0) or a
 * non-zero status and never aborts; pgxc_last_error() describes the failure,
 * which the Fortran caller routes to error_handler (error_handler.f90), as
 * ASSERT/ABORT do in the reference (include/def.h:10-18).
 *
 * Threading: one context = one HIP stream on the current device.  A context is
 * not re-entrant; distinct contexts share no state.
 */
#ifndef PGXC_H
#define PGXC_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* status codes */
#define PGXC_OK 0
#define PGXC_ERR_ARG 1         /* invalid argument or shape                   */
#define PGXC_ERR_UNSUPPORTED 2 /* functional / spin / l not supported          */
#define PGXC_ERR_HIP 3         /* HIP runtime error (message says which call)  */
#define PGXC_ERR_NOMEM 4       /* device allocation failed                    */
#define PGXC_ERR_STATE 5       /* call out of order (e.g. build before density) */

/* Functional terms: bit (1 << e) for each enabled xc_cntrl enumerator e
 * (modules/xc_cntrl.f90:61-104).  Terms are summed in enum order with
 * frac = 1 (modules/xc_func.f90:284-304).  XC="PBE" selects all four
 * (modules/xc_cntrl.f90:652-670). */
#define PGXC_XC_XALPHA (1u << 1)
#define PGXC_XC_PWLDAC (1u << 3)
#define PGXC_XC_PBEX (1u << 10)
#define PGXC_XC_PBEC (1u << 18)
#define PGXC_XC_LDA (PGXC_XC_XALPHA | PGXC_XC_PWLDAC)
#define PGXC_XC_PBE (PGXC_XC_XALPHA | PGXC_XC_PWLDAC | PGXC_XC_PBEX | PGXC_XC_PBEC)

/* Arithmetic of the two contractions (Phi P and Phi^T W).  The functional,
 * per-point state, E_xc/charge and V accumulation are FP64 in every mode;
 * basis values are evaluated and stored in FP64 for FP64 builds and in FP32
 * for both mixed modes (centre offsets formed in FP64 first). */
#define PGXC_PREC_FP64 0   /* FP64 MFMA                                     */
#define PGXC_PREC_FP32 1   /* FP32 MFMA, FP32 accumulation                   */
#define PGXC_PREC_BF16X3 2 /* split-BF16 (hi*hi + hi*lo + lo*hi), FP32 acc.  */

/* density modes for pgxc_set_density / pgxc_set_orbitals */
#define PGXC_DENSITY_FULL 0        /* next build integrates P itself          */
#define PGXC_DENSITY_INCREMENTAL 1 /* next build integrates dP = P - P_prev   */

/* Schedules of the two contraction stages (pgxc_set_schedule,
 * pgxc_batch_set_schedule).  They change which workgroup computes which work
 * item and when, never a result bit. */
#define PGXC_SCHED_STATIC 0   /* fixed round-robin walk                        */
#define PGXC_SCHED_ANALYTIC 1 /* queues balanced by counted flops (the default) */
#define PGXC_SCHED_MODEL 2    /* queues balanced by the cost model's prediction */

/* Features of one work item, in this order (pgxc_item_log, cost model):
 * kind (0 density, 1 potential contraction), precision one-hot (FP64, FP32,
 * BF16x3), columns / 128 (density: the share of its tile's functions that an
 * item takes, in whole blocks of 16; potential: the functions of a chunk),
 * log2(1 + K length left after screening) / 16, log2(1 + dense K length) / 16,
 * 1 if any block is left after screening, variant / 2.  (K: functions of the
 * density contraction, in whole runs of 8 for BF16x3; points of the potential
 * contraction.) */
#define PGXC_NFEATURES 9

typedef struct pgxc_ctx pgxc_ctx;
typedef struct pgxc_batch pgxc_batch;
typedef struct pgxc_costmodel pgxc_costmodel;

/* Layout options of a context (pgxc_create_opt).  tile: 64, 96 or 128: nbas is
 * padded to a multiple of it, and the potential contraction takes its functions
 * in chunks of it (0: the padding is the least of the three, the chunks follow
 * the functions a point split has).
 * chunk_points: largest number of grid points held in one work chunk, a
 * multiple of 2048 (0: at most 256 Ki points and 8 GiB of FP64 basis values).
 * variant_fp64 / variant_fp32: contraction kernel variant for FP64 and FP32
 * builds, 0 (K step 16, two LDS stages), 1 (K step 32, one LDS stage),
 * 2 (K step 32, two LDS stages); -1 keeps the default.  pgxc/autotune.py picks
 * tile and variants by timing them.  no_screen: 1 runs the contractions over
 * every basis function and point; 0 (default) leaves out, per tile of 128
 * points, the shells whose every value there the radial cut-off
 * alpha r^2 >= 50 (modules/orbital_module.f90:1839-1855) makes exactly zero:
 * only the rounding of the regrouped sums differs.  no_basis_cache: 1 evaluates the
 * basis values in every build; 0 (default) keeps the values of every grid
 * chunk on the device after the first build of each precision and reuses
 * them (the role of ParaGauss's orbital store across SCF cycles,
 * modules/orbitalstore_module.f90:862-977), when they fit in a quarter of the
 * device memory. */
typedef struct pgxc_options {
  int32_t tile;
  int64_t chunk_points;
  int32_t variant_fp64;
  int32_t variant_fp32;
  int32_t no_screen;
  int32_t no_basis_cache;
} pgxc_options;

/*
 * Create a context on the current HIP device.
 *
 * Basis (C1, the order of modules/orbitalprojection_module.f90:30-50):
 *   shell_info[5*s .. 5*s+4] = atom, l, n_exp, n_unc, n_contr for shell s
 *     (one shell per (unique atom, l), as unique_atom_basis_type,
 *      modules/unique_atom_module.f90:143-168).  A shell yields
 *      (2l+1)*(n_unc+n_contr) functions, m outer, radial function inner
 *      (modules/orbital_module.f90:2509-2610).
 *   exps, norms: concatenated per shell (n_exp each); norms as
 *      unique_atom_basis_norm_ob (modules/unique_atom_module.f90:426-444).
 *   contr: concatenated per shell, n_exp x n_contr column-major each.
 *   atom_xyz: 3 doubles per atom (bohr).
 * Grid: grid is npts x 4 column-major (x, y, z, w), the layout of grdpts
 *   (modules/grid_module.f90:194,3093).  The reference integrates contiguous
 *   veclen-point batches in grid order (more_grid,
 *   modules/grid_module.f90:1133-1181; veclen = machineparameters_veclen,
 *   default 128); the library regroups the points along a space-filling curve
 *   so that its point tiles are compact in space.  Every result is a sum over
 *   points, so only the rounding of the sums depends on the grouping.
 * Replaces: the setup part of xc_build (xc_allocate/orbital_setup,
 *   modules/xc_hamiltonian.f90:239-283) plus the device upload of grid/basis.
 */
int pgxc_create(pgxc_ctx **ctx, int32_t n_atoms, const double *atom_xyz,
                int32_t n_shells, const int32_t *shell_info, const double *exps,
                const double *norms, const double *contr, const double *grid,
                int64_t npts, int32_t veclen);

/* pgxc_create with layout options (opt may be NULL).  No counterpart in the
 * reference: the batch path (pgxc_batch_*) uses it to size many contexts. */
int pgxc_create_opt(pgxc_ctx **ctx, int32_t n_atoms, const double *atom_xyz,
                    int32_t n_shells, const int32_t *shell_info, const double *exps,
                    const double *norms, const double *contr, const double *grid,
                    int64_t npts, int32_t veclen, const pgxc_options *opt);

/* Layout chosen for a context: [0] padded nbas, [1] function tile,
 * [2] points per chunk, [3] chunks, [4] blocks of 2048 or more points a chunk
 * is made of (the potential contraction cuts them into shorter splits),
 * [5] padded number of points, [6] FP64 variant, [7] FP32 variant. */
int pgxc_layout(const pgxc_ctx *ctx, int64_t *out8);

/*
 * Density matrix P (nbas x nbas x ispin, column-major, symmetric): the total
 * density for ispin = 1; the alpha then the beta spin's for ispin = 2
 * (rho(vl, ispin) of modules/density_calc_module.f90:1478-1577).  Equivalent
 * to eigvec_occ / occ_num_occ (modules/occupied_levels_module.f90:112-117)
 * through P_s = C_s diag(occ_s) C_s^T.  mode = PGXC_DENSITY_INCREMENTAL makes
 * the next build integrate dP against the state left by the previous build
 * on this context (same ispin, else PGXC_ERR_STATE); a full density with
 * another ispin than the last one drops that state.
 */
int pgxc_set_density(pgxc_ctx *ctx, int32_t ispin, int32_t nbas, const double *P,
                     int32_t mode);

/* Occupied orbitals C (nbas x nocc x ispin, column-major) and occupations
 * occ (nocc x ispin), exactly the arguments density_calc_nl reads
 * (eigvec_occ(irr)%m(N, n_occ, ispin), occ_num_occ(irr)%m(n_occ, ispin),
 * modules/density_calc_module.f90:1490-1540); P is formed on the device. */
int pgxc_set_orbitals(pgxc_ctx *ctx, int32_t ispin, int32_t nbas, int32_t nocc,
                      const double *C, const double *occ, int32_t mode);

/*
 * One XC build over all batches.  Replaces the body of calc_xcks_nl (GGA) /
 * calc_xcks (LDA).  ham_packed has ispin*nbas*(nbas+1)/2 doubles and receives
 * ham_xc_arr ADDED INTO (the reference accumulates into the zeroed array,
 * modules/xc_hamiltonian.f90:1561-1567); packing (j = 1..n, k = 1..j), for
 * ispin = 2 the alpha and beta spins interleaved at even / odd positions
 * (counter = s, step ispin, :1455-1460).
 * exc and charge are also added into (exc_int, charge_int, :1408,1423).
 * Any of ham_packed / exc / charge may be NULL to leave the result on the
 * device (pgxc_get_result fetches it).
 */
int pgxc_build(pgxc_ctx *ctx, uint32_t functional, int32_t precision,
               double *ham_packed, double *exc, double *charge);

/* Copy the last build's results (same semantics as pgxc_build's outputs). */
int pgxc_get_result(pgxc_ctx *ctx, double *ham_packed, double *exc, double *charge);

/*
 * XC energy of each functional term on the current density, without the
 * potential matrix: the post-SCF energy evaluation of post_scf_calc_xc_energy
 * (modules/post_scf_module.f90:2204-2420), which integrates every enabled
 * functional's energy on the converged density.  terms4 receives (written,
 * not added) the energies of XAlpha, PWLDAc, PBEx and PBEc (0 for a term not
 * in the mask; PBEx and PBEc are the gradient corrections, so the PBE energy
 * is their sum with the first two), charge the integrated density.  Uses the
 * full density of the last pgxc_set_density / pgxc_set_orbitals (either
 * ispin) and runs only the basis, density and functional stages; the state of
 * incremental builds and the last build's results are left as they are.
 */
int pgxc_energy(pgxc_ctx *ctx, uint32_t functional, int32_t precision, double *terms4,
                double *charge);

/*
 * Nuclear gradient of E_xc, the basis-centre term F1 of post_scf_module
 * (modules/post_scf_module.f90:150-185: -2 sum P_ij <d/dR xi_i | V_xc | xi_j>,
 * summed over spins), which is grad_xc when weight_grads is off; the grid
 * and its weights are held fixed (the weight-derivative term F2 is not
 * computed).  grad (n_atoms x 3, row-major by atom, caller atom order)
 * receives dE_xc/dR (written, not added; the reference stores the negative).
 * Evaluated at the density matrix and potential coefficients of the last
 * build on the context, in FP64 whatever that build's precision: the basis
 * and its second derivatives per point, and two products with P on the
 * screened tiles.  The first call allocates the work space of one chunk (the
 * products, 16 bytes per function and point of a chunk, and the sums' parts)
 * and the context keeps it.
 */
int pgxc_gradient(pgxc_ctx *ctx, double *grad);

/*
 * The full nuclear gradient of E_xc with the grid moving with the atoms
 * (weight_grads on, the reference's default, modules/grid_module.f90:240-245):
 * F1 + F2 of modules/post_scf_module.f90:150-172, F2 = sum_a dw_a/dR e_xc(r_a)
 * + sum_a w_a dr_a/dR . grad e_xc(r_a) for Becke-partitioned weights (no
 * atomic-size adjustment) of points that move rigidly with their owner atom.
 * owner[npts] (caller point order): the atom whose atomic grid holds the
 * point; the grid's weights must be the Becke partition of those atomic
 * grids.  grad (n_atoms x 3) receives dE_xc/dR, at the last build's density
 * and coefficients, FP64.  The first call allocates 40 bytes per point, 8 per
 * pair of atoms and at most 256 MiB of scratch, which the context keeps.
 */
int pgxc_gradient_grid(pgxc_ctx *ctx, const int32_t *owner, double *grad);

/* Number of basis functions of the context (dims(1) in C1). */
int64_t pgxc_nbas(const pgxc_ctx *ctx);

/* Work counters of the last build: [0] points, [1] batches, [2] algorithmic
 * flops (4 B n^2 + 16 B n summed over 128-point batches, n = screened
 * functions, times ispin), [3] exp evaluations, [4] HBM bytes of the
 * algorithmic model: the same sum of 32 B (x, y, z, w) + 16 n^2 ispin (P
 * sub-block read, V partial written) + 4 s B n (basis values and gradients
 * at s = 8 bytes in FP64 builds, 4 in FP32 and split-BF16 builds). */
int pgxc_last_stats(const pgxc_ctx *ctx, double *stats5);

/* The screened sizes behind those counters (no counterpart in the
 * reference): [0] sum over 128-point batches of B n (points times screened
 * functions), [1] sum of n^2, [2] number of batches. */
int pgxc_last_work(const pgxc_ctx *ctx, double *work3);

/* Device timing of the last build's kernels in milliseconds, by stage:
 * [0] basis, [1] density contraction, [2] functional, [3] potential
 * contraction, [4] reductions/packing, [5] whole build. */
int pgxc_last_timing(const pgxc_ctx *ctx, double *ms6);

/* Message of the context's last failure; with ctx = NULL, that of the last
 * failed context-free call (pgxc_becke_weights_noalloc). */
const char *pgxc_last_error(const pgxc_ctx *ctx);

/*
 * Grid generation: Becke partition of atom-centred one-centre weights.
 * Replaces becke0 (modules/grid_module.f90:2442-2497) with the step function
 * mu3 = p(p(p(mu))) (autodiff/becke_step_func.f90:84-124), atomic-size
 * adjustment off (art = 0, modules/grid_module.f90:2344-2347).
 *   pts: npts x 3 column-major; owner[p]: atom hosting point p;
 *   w_atomic[p]: its one-centre weight w_ang * w_rad * 4 pi
 *   (modules/grid_module.f90:426-433); w_out[p] = w_atomic[p] * P_owner / sum_i P_i.
 * Context-free; runs on the current device.
 */
int pgxc_becke_weights(int32_t n_atoms, const double *atom_xyz, int64_t npts,
                       const double *pts, const int32_t *owner, const double *w_atomic,
                       double *w_out);

/*
 * pgxc_becke_weights without any device allocation.  No counterpart in the
 * reference: for callers that cannot allocate device memory (code under HIP
 * graph capture, serving loops, harnesses that forbid hipMalloc).  Every
 * array is DEVICE memory the caller owns, in pgxc_becke_weights' layouts:
 * atom_xyz (3 per atom), pts (npts x 3 column-major), owner, w_atomic and
 * w_out (npts each).  The work is queued on stream (a hipStream_t of the
 * current device; NULL: the default stream) and the call returns without
 * waiting; w_out then holds the bits pgxc_becke_weights gives.  The table of
 * inverse pair distances lives in a file-scope device array of 1024 x 1024
 * doubles (8 MiB on each device that runs the call, held until the process
 * ends): n_atoms above 1024 is refused with PGXC_ERR_ARG, and
 * pgxc_last_error(NULL) says why.  Calls that overlap on one device share
 * that array and race: order them on one stream.  An owner out of range
 * gives weight 0 and coincident centres give NaN (pgxc_becke_weights reports
 * both as PGXC_ERR_ARG).
 */
int pgxc_becke_weights_noalloc(int32_t n_atoms, const double *atom_xyz, int64_t npts,
                               const double *pts, const int32_t *owner, const double *w_atomic,
                               double *w_out, void *stream);

int pgxc_destroy(pgxc_ctx *ctx);

/*
 * Batches: the XC builds of many molecules (contexts, each with its own
 * basis, grid and density) run together, one launch per stage over the work
 * items of all of them, optionally replayed from a captured hipGraph.  In the
 * reference every molecule is a separate ParaGauss run; the batch replaces that
 * loop of xc_build calls.  Each context keeps its own results
 * (pgxc_get_result) and incremental state, exactly as after pgxc_build.
 * Results do not depend on the schedule: every work item writes its own
 * partial sums, reduced in a fixed order.  Every context keeps its own work
 * memory while it lives: a chunk's W and (uncached) basis values per lane, the
 * potential's partial sums (those of all its chunks, up to 4 GiB per spin) and
 * 2 MiB of pinned host memory; a smaller chunk_points makes the first smaller.
 */
int pgxc_batch_create(pgxc_batch **batch, int32_t n, pgxc_ctx *const *ctxs);

/* Schedule priority per molecule (n doubles, e.g. predicted cost; larger runs
 * first); NULL restores the natural order. */
int pgxc_batch_set_priority(pgxc_batch *batch, const double *cost);

/* One build of every molecule; use_graph = 1 captures the launch sequence
 * into a hipGraph on first use and replays it afterwards. */
int pgxc_batch_build(pgxc_batch *batch, uint32_t functional, int32_t precision,
                     int32_t use_graph);

/* Device time of the last batch build (ms). */
int pgxc_batch_last_ms(const pgxc_batch *batch, double *ms);

const char *pgxc_batch_last_error(const pgxc_batch *batch);

int pgxc_batch_destroy(pgxc_batch *batch);

/*
 * Work distribution and the learned cost model.
 *
 * The reference hands each MPI rank a static contiguous share of the grid
 * batches (distribute_jobs, dlb/dlb_common.f90:516-561, through dlb_setup /
 * dlb_give_more, dlb/dlb.f90:203-224,290-311).  Here the work items of a
 * contraction launch (point tile x function tile, or point split x function
 * tile pair) are either walked round-robin (PGXC_SCHED_STATIC), or cut into
 * one queue per XCD of about equal predicted cost, each ordered costliest
 * first, and drained dynamically (a workgroup whose queue is empty takes from
 * the next) (PGXC_SCHED_ANALYTIC: counted flops left after screening;
 * PGXC_SCHED_MODEL: the cost model).  The model is a 3-layer MLP
 * (PGXC_NFEATURES -> 64 -> 64 -> 1, tanh) predicting log(item time / us),
 * trained on the GPU from the per-item timings this library logs.  The
 * context (batch) keeps the model pointer: the model must outlive it, or the
 * schedule must be changed before the model is destroyed.
 */
int pgxc_set_schedule(pgxc_ctx *ctx, int32_t mode, pgxc_costmodel *model);
int pgxc_batch_set_schedule(pgxc_batch *batch, int32_t mode, pgxc_costmodel *model);

/*
 * State of incremental builds, for checkpoint / restart.  The reference
 * saves ham_xc_arr and exc_int to its SCF state file
 * (xc_hamiltonian_store / xc_hamiltonian_recover,
 * modules/xc_hamiltonian.f90:2407-2633); those records are unchanged here.
 * The library's own state between builds (the previous density matrix, the
 * packed V of the last build and the FP64 per-point density and potential
 * coefficients) is what an incremental build continues from: saving it
 * beside those records lets a restarted SCF continue with incremental builds
 * that give the same bits as without the restart.  pgxc_state_bytes: size of
 * the record.  pgxc_save_state: needs a build on the context.
 * pgxc_load_state: only into a context of the same atoms, basis, grid and
 * layout (checked by a hash recorded in the state); PGXC_ERR_ARG otherwise.
 * The record holds every spin of the build (ispin = 2: twice the size) and
 * loading it sets the context's ispin, which the next (incremental) density
 * must then use.
 */
int64_t pgxc_state_bytes(const pgxc_ctx *ctx);
int pgxc_save_state(pgxc_ctx *ctx, void *buf, int64_t bytes);
int pgxc_load_state(pgxc_ctx *ctx, const void *buf, int64_t bytes);

/* Lanes of later builds (no counterpart in the reference: the reference's
 * batches run one after another on one CPU core).  A grid of more than one
 * chunk is built on two lanes by default: chunk k runs on stream k % 2 with
 * its own work buffers, so one chunk's stages overlap the next chunk's.
 * lanes = 1 runs every chunk on one stream (each launch then has the device
 * to itself, which is how per-kernel timings are measured); 2 restores the
 * default.  Results agree to rounding (the H partials are summed per lane).
 * A batch runs two lanes only when every member of more than one chunk has
 * two; otherwise all of its members run on one lane, and each member's
 * results are the bits of its own build at that lane count. */
int pgxc_set_lanes(pgxc_ctx *ctx, int32_t lanes);

/* on = 1: later builds record, per contraction work item, its features and
 * the device time its workgroup spent on it. */
int pgxc_set_item_log(pgxc_ctx *ctx, int32_t on);
int pgxc_batch_set_item_log(pgxc_batch *batch, int32_t on);

/* Items of the last logged build: returns their number n (negative on
 * error); when cap >= n, features (n x PGXC_NFEATURES, row-major) and us
 * (n) are filled. */
int64_t pgxc_item_log(pgxc_ctx *ctx, double *features, double *us, int64_t cap);
int64_t pgxc_batch_item_log(pgxc_batch *batch, double *features, double *us, int64_t cap);

/* Cost model with n_features inputs, Glorot-uniform weights from seed. */
int pgxc_costmodel_create(pgxc_costmodel **model, int32_t n_features, uint64_t seed);

/* Number of parameters: F*64 + 64 + 64*64 + 64 + 64 + 1, flat in the order
 * W1[F][64], b1, W2[64][64], b2, w3, b3. */
int32_t pgxc_costmodel_nparams(const pgxc_costmodel *model);

/* Parameters (nparams) and, if norm is not NULL, the standardisation
 * (2 F + 2: feature means, feature scales, target mean, target scale). */
int pgxc_costmodel_params(pgxc_costmodel *model, double *params, double *norm);
int pgxc_costmodel_set_params(pgxc_costmodel *model, const double *params, const double *norm);

/* steps full-batch Adam steps (learning rate lr) on the mean squared error
 * of the standardised targets y (n) from features X (n x F, row-major); the
 * first training call fixes the standardisation.  loss (optional): the final
 * loss. */
int pgxc_costmodel_train(pgxc_costmodel *model, const double *X, const double *y, int64_t n,
                         int32_t steps, double lr, double *loss);

/* Gradient (nparams) of that loss at the current parameters, and the loss. */
int pgxc_costmodel_gradient(pgxc_costmodel *model, const double *X, const double *y, int64_t n,
                            double *grad, double *loss);

/* Predictions (n, in the target's units) for features X (n x F). */
int pgxc_costmodel_predict(pgxc_costmodel *model, const double *X, int64_t n, double *out);

const char *pgxc_costmodel_last_error(const pgxc_costmodel *model);

int pgxc_costmodel_destroy(pgxc_costmodel *model);

#ifdef __cplusplus
}
#endif
#endif /* PGXC_H */
