/*
 * gpstep.h -- C ABI of the MI355X grand-potential 2-D finite-difference step.
 *
 * Drop-in for the time-loop body of the MicroSim serial grand-potential solver
 * (Grand_potential_Finite_difference_2D_serial):
 *
 *     solverloop_phasefield(start,end);   apply_boundary_conditions(0);
 *     solverloop_concentration(start,end); apply_boundary_conditions(0);
 *
 * (microsim_gp.c:103-106).  In the reference all data travels through globals
 * (functions/global_vars.h); here it travels through a gp_params block of
 * host-derived constants and an opaque context that owns the device fields.
 *
 * Conventions
 *   - P = NUMPHASES (the last phase, P-1, is the liquid / reference phase),
 *     C = NUMCOMPONENTS-1 independent diffusion potentials.
 *   - Host-side field arrays are interior-only, planar, x-major with y fastest:
 *       phi[a][x][y] = phi[(a*mesh_x + x)*mesh_y + y],  a < P
 *       mu [k][x][y] = mu [(k*mesh_x + x)*mesh_y + y],  k < C
 *     which is the order of the reference's VTK blocks (file_writer.h:86-111).
 *   - Every entry point returns 0 on success or a negative GP_E_* code; no entry
 *     point exits the process.  gp_strerror() names the code.
 *   - Contexts share nothing; calls on different contexts may run concurrently
 *     from different host threads.
 */
#ifndef GPSTEP_H_
#define GPSTEP_H_

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define GP_MAX_PHASES 16   /* P limit of the parameter block               */
#define GP_MAX_COMP   4    /* C limit (NUMCOMPONENTS-1) of the parameter block */

/* error codes */
#define GP_OK              0
#define GP_E_ARG          -1   /* bad argument / inconsistent parameters         */
#define GP_E_UNSUPPORTED  -2   /* valid input that this build does not implement */
#define GP_E_HIP          -3   /* HIP runtime error                              */
#define GP_E_NOMEM        -4   /* host or device allocation failed               */
#define GP_E_NONFINITE    -5   /* non-finite value found in the fields           */
#define GP_E_IO           -6   /* file could not be opened / parsed              */
#define GP_E_NODEVICE     -7   /* no HIP device visible                          */
#define GP_E_SCRATCH      -8   /* grid too large for the no-allocation scratch   */

/* chemical-potential update flavour (calculate_divergence_concentration.h:93-125) */
#define GP_MU_GENERAL  0   /* LU inverse of dc/dmu (matrix.h:50-114)  */
#define GP_MU_BINARY   1   /* scalar 1/dcdmu                          */
#define GP_MU_TERNARY  2   /* closed-form 2x2 inverse                 */
#define GP_MU_DILUTE   3   /* diagonal inverse                        */

/* boundary types (utility_functions.h:471-653): 0 free, 1 Neumann, 2 Dirichlet, 3 periodic */
#define GP_BC_FREE      0
#define GP_BC_NEUMANN   1
#define GP_BC_DIRICHLET 2
#define GP_BC_PERIODIC  3

/* faces, in the reference's boundary[] numbering */
#define GP_FACE_XMIN 0
#define GP_FACE_XMAX 1
#define GP_FACE_YMAX 2
#define GP_FACE_YMIN 3

/* data types of a context */
#define GP_F64 0   /* bulk stencil in binary64 (parity path)                     */
#define GP_F32 1   /* bulk stencil in binary32, compensated mu, FP64 reductions  */

/*
 * Parameter block: everything one step reads.  The tables hold the values the
 * reference keeps in globals after reading_input_parameters() and
 * init_propertymatrices(T) (functions/functionF_01.h:169-230); gp_derive() in
 * gpio.h fills the derived ones from the raw ones.  Unused entries must be 0.
 */
typedef struct gp_params {
  long   mesh_x, mesh_y;          /* MESH_X, MESH_Y (interior cells)              */
  double dx, dy, dt;              /* DELTA_X, DELTA_Y, DELTA_t                    */
  int    nphases;                 /* P                                            */
  int    ncomp;                   /* C = NUMCOMPONENTS-1                          */
  int    obstacle;                /* 1: obstacle potential (Function_W=1), 0: well (Function_W=2) */
  int    anisotropy;              /* Function_anisotropy: 0 isotropic, 1 four-fold cubic */
  int    mu_solver;               /* GP_MU_*                                      */
  int    isothermal;              /* ISOTHERMAL (0: temperature gradient in y, below) */
  double epsilon;                 /* interface width parameter                    */
  double tau;                     /* scalar relaxation constant (functionTau.h:13) */
  double T, Teq;                  /* temperature, equilibrium temperature         */
  /* ghost-layer copies: bc_type[field][face], field 0 = phi, 1 = mu; proxy[field][face][j]
     is the padded index copied into ghost layer points[face][j] (assign_boundary_points_values) */
  int    bc_type[2][4];
  long   bc_proxy[2][4][3];
  /* phase-pair tables */
  double gamma[GP_MAX_PHASES][GP_MAX_PHASES];                     /* GAMMA        */
  double gamma_abc[GP_MAX_PHASES][GP_MAX_PHASES][GP_MAX_PHASES];  /* Gamma_abc    */
  double tau_ab[GP_MAX_PHASES][GP_MAX_PHASES];                    /* Tau          */
  double dab[GP_MAX_PHASES][GP_MAX_PHASES];                       /* dab          */
  double rot[GP_MAX_PHASES][GP_MAX_PHASES][3][3];                 /* Rotation_matrix (after inversion) */
  double rot_inv[GP_MAX_PHASES][GP_MAX_PHASES][3][3];             /* Inv_Rotation_matrix */
  /* thermodynamic tables */
  double diffusivity[GP_MAX_PHASES][GP_MAX_COMP][GP_MAX_COMP];    /* DIFFUSIVITY  */
  double A[GP_MAX_PHASES][GP_MAX_COMP][GP_MAX_COMP];              /* A            */
  double ceq[GP_MAX_PHASES][GP_MAX_PHASES][GP_MAX_COMP];          /* ceq          */
  double cfill[GP_MAX_PHASES][GP_MAX_PHASES][GP_MAX_COMP];        /* cfill        */
  double slopes[GP_MAX_PHASES][GP_MAX_PHASES][GP_MAX_COMP];       /* slopes       */
  /* derived by gp_derive() */
  double cmu[GP_MAX_PHASES][GP_MAX_COMP][GP_MAX_COMP];            /* (dmu/dc)^-1  */
  double Beq[GP_MAX_PHASES][GP_MAX_COMP];
  double dBbdT[GP_MAX_PHASES][GP_MAX_COMP];
  double B[GP_MAX_PHASES][GP_MAX_COMP];                           /* B(T)         */
  double Cf[GP_MAX_PHASES];                                       /* C(T)         */
  /* derived by gp_derive(): DELTA_T[a][a], DELTA_T[a][liquid] and DELTA_C[a] of
     each solid (functionF_01.h:195-205), for B(T) and C(T) of other temperatures */
  double delta_T_s[GP_MAX_PHASES], delta_T_l[GP_MAX_PHASES];
  double delta_C[GP_MAX_PHASES][GP_MAX_COMP];
  /* non-isothermal runs (isothermal = 0): the temperature is linear in y,
     temp_bottom + y*DeltaT*dy/Distance, and moves with the velocity
     (functions/Temperature_gradient.h:4-29, microsim_gp.c:77-113) */
  double tempgrad[5];             /* Tempgrady = {base_temp, DeltaT, Distance, gradient_OFFSET, velocity} */
  int    bc_type_T[4];            /* BOUNDARY = {T, ...} types; 0: the ghost layers are not copied */
  long   bc_proxy_T[4][3];        /* padded index copied into each temperature ghost layer */
  /* phase-field noise (Noise_phasefield, Amp_Noise_Phase): the phase sweep adds
     amp_noise * rand()/RAND_MAX * phi_a (1 - phi_a) to lambda_a of every active
     phase, drawing glibc rand() in the serial sweep order
     (solverloop/calculate_divergence_phasefield.h:33-34); a context starts the
     sequence as an unseeded process does (srand(1), gp_noise_seed) */
  int    noise;
  double amp_noise;
  /* F_01 semantics of the reference's MPI solver as options (GP_MPI_* bits;
     0: the serial solver), run on the two-pass path in binary64 */
  int    mpi;
  double V;                       /* V (molar volume): GP_MPI_TAU, GP_MPI_DPSI_V */
  unsigned long long mpi_rand;    /* drand48 state (48 bits) before the first
                                     step's draws (GP_MPI_NOISE); an unseeded
                                     process starts at 0x1234ABCD330E */
} gp_params;

/* MPI solver semantics (Grand_potential_Finite_difference_2D_MPI, one worker,
   whose padded grid is the serial one: solverloop/mpiinfo_xy.h:195-224):
   GP_MPI_COMPOSITION  a composition field c is carried: every cell adds
                       dt div(M grad mu) - div(j_at) to c, and a cell with
                       phi_a == 1 takes mu = Mu_a(c) instead of the serial
                       c_a(mu) round trip; interface cells keep the serial mu
                       update (calculate_divergence_concentration.h:379-545)
   GP_MPI_TAU          Calculate_Tau replaces Tau: tau_aL = (dmu . dc) eps
                       0.2222 / V per solid, its minimum elsewhere
                       (functionTau.h:18-54, microsim_gp.c:149-150)
   GP_MPI_DPSI_V       lambda takes -dpsi/V (calculate_divergence_phasefield.h:339)
   GP_MPI_NOISE        with noise: one drand48() draw per cell of the phase
                       sweep, lambda_a += 4 AMP r phi_a (1 - phi_a) dpsi / V
                       (calculate_divergence_phasefield.h:335-343)
   GP_MPI_YSKIP        the y-face antitrapping skip sits at end[Y]+2 = MESH_Y+4,
                       a ghost row, so no interior face is skipped
                       (calculate_fluxes_concentration.h:209)
   GP_MPI_GHOST_DPHI   the boundary copies after the phase sweep copy
                       delta-phi too, so ghost delta-phi = its source's
                       (boundary_mpi.h:94-105) */
#define GP_MPI_COMPOSITION 1
#define GP_MPI_TAU         2
#define GP_MPI_DPSI_V      4
#define GP_MPI_NOISE       8
#define GP_MPI_YSKIP       16
#define GP_MPI_GHOST_DPHI  32
#define GP_MPI_ALL         63
#define GP_DRAND48_SEED    0x1234ABCD330EULL

/* Global diagnostics of the current state (replaces the TRACK_PROGRESS print of
   microsim_gp.c:139-148, restricted to interior cells; sums in binary64). */
typedef struct gp_stats {
  double phi_max[GP_MAX_PHASES], phi_min[GP_MAX_PHASES];
  double mu_max[GP_MAX_COMP],    mu_min[GP_MAX_COMP];
  double phi_sum[GP_MAX_PHASES];            /* sum of phi_a over interior cells          */
  double solute[GP_MAX_COMP];               /* sum_cells w * sum_a h_a(phi) c_a(mu)       */
  double nonfinite;                         /* number of non-finite interior values      */
  double rel_change_phi[GP_MAX_PHASES];     /* sum of (change of phi_a in the last step)^2 */
  double rel_change_mu[GP_MAX_COMP];        /* sum of (change of mu_k in the last step)^2  */
  /* Free-energy functional in binary64, summed over interior nodes with the
     solute sum's weights and times dx dy.  The reference's phase sweep is its
     variational derivative; the reference itself never sums it.  */
  double energy_gradient;                   /* eps a(phi, grad phi)                       */
  double energy_potential;                  /* w(phi) / eps                               */
  double energy_bulk;                       /* sum_a h_a(phi) psi_a(mu, T)                */
  double grand_potential;                   /* the three terms above                      */
  double free_energy;                       /* grand_potential + sum_k mu_k c_k           */
} gp_stats;

typedef struct gp_ctx gp_ctx;

/* Create a context: validates p, copies it to the device, allocates the fields.
   dtype is GP_F64 or GP_F32.  Replaces serialinfo_xy() + the allocation part of
   main() (microsim_gp.c:43-47, solverloop/serialinfo_xy.h:1-66). */
int  gp_create(const gp_params *p, int dtype, gp_ctx **out);
void gp_destroy(gp_ctx *ctx);

/* Load / read back the interior fields (host arrays in the layout above, binary64).
   gp_set_state also fills the ghost layers, like apply_boundary_conditions(0)
   after fill_domain / restart reading (microsim_gp.c:48-57,84).  The fields
   pass through P + C binary64 planes of device memory: a context that needs at
   most GP_TRANSIT_KEEP bytes for them keeps them from its first call until it is
   destroyed; a larger one gives them back before the call returns. */
#define GP_TRANSIT_KEEP (8u << 20)
int  gp_set_state(gp_ctx *ctx, const double *phi, const double *mu);
int  gp_get_state(gp_ctx *ctx, double *phi, double *mu);

/* Composition field of a context with GP_MPI_COMPOSITION (interior planar
   [C][MESH_X][MESH_Y], binary64).  gp_set_state and gp_set_state_device set
   it to sum_a h_a(phi) c_a(mu) per cell; gp_set_composition replaces it (the
   MPI fill gives bulk cells ceq / cfill exactly, fill_composition_cube of
   MPI functions/filling.h:876-925).  GP_E_UNSUPPORTED without the field.
   Replaces the composition member of the MPI solver's struct fields. */
int  gp_set_composition(gp_ctx *ctx, const double *comp);
int  gp_get_composition(gp_ctx *ctx, double *comp);
/* drand48 state of the MPI noise after the steps run so far (48 bits);
   GP_E_UNSUPPORTED unless GP_MPI_NOISE and noise are set. */
int  gp_get_rand_state(gp_ctx *ctx, unsigned long long *state);

/* Same, with device pointers of the context's dtype (float or double) holding the
   interior layout above; ordered on the context's stream. */
int  gp_set_state_device(gp_ctx *ctx, const void *phi, const void *mu);
int  gp_get_state_device(gp_ctx *ctx, void *phi, void *mu);

/* Advance nsteps explicit Euler steps: each step is the phase sweep, ghost copy,
   concentration sweep and ghost copy of microsim_gp.c:103-106. */
int  gp_step(gp_ctx *ctx, long nsteps);

/* Wait for all work of the context (host-side timing without another runtime). */
int  gp_synchronize(gp_ctx *ctx);

/* nsweeps pre-loop smoothing sweeps (the NSMOOTH-1 calls of smooth() and the
   ghost copies, microsim_gp.c:97-100; solverloop/solverloop.h:72-90). */
int  gp_smooth(gp_ctx *ctx, long nsweeps);

/* Diagnostics of the current state. */
int  gp_stats_get(gp_ctx *ctx, gp_stats *st);

/* Stream the context enqueues on (a hipStream_t; NULL = the default stream). */
int  gp_set_stream(gp_ctx *ctx, void *hip_stream);

/* Device-side time of the last gp_step call in milliseconds (hipEvents on the
   context's stream, bracketing every kernel of that call). */
int  gp_last_step_ms(gp_ctx *ctx, double *ms);

/* Kernel path of a context: 0 = fused LDS kernel on interface tiles plus a
   diffusion-only kernel on bulk tiles, 1 = two-pass kernels (phase
   kernel + concentration kernel over the whole grid), 2 = fused LDS kernel on
   every tile, 3 = two-pass kernels on interface tiles (cells sorted in LDS into
   interface and bulk cells) plus the bulk kernel, 4 = split two-pass: per sweep
   a light kernel finishes the bulk cells and lists the blocks holding others,
   which the two-pass kernels then update, 5 = compact split: as 4, but the
   light kernels list the cells themselves and the dense kernels run one listed
   cell per lane, 6 = one-hot: as 5, with a byte per cell and state buffer
   recording where that buffer holds an exact one-hot phase vector, so that
   bulk cells are classified and updated without loading their phase fields
   and their unchanged phase fields are not written again, and with the dense
   phase sweep and the light mu sweep in one launch, -1 = automatic (the
   default): at the start, after 64 blocks of 32 steps and then at doubling
   gaps, one block of each of paths 1, 4, 5 and 6 is timed (as graph replays,
   or as direct launches where graphs are off) and the fastest runs until the
   next re-timing.  All paths give bit-identical binary64 results.
   Non-isothermal and noise contexts step on paths 1, 4, 5 and 6 only (other
   values: GP_E_UNSUPPORTED). */
int  gp_set_path(gp_ctx *ctx, int path);
/* The path in use (after automatic choices) and whether the choice is automatic. */
int  gp_get_path(gp_ctx *ctx, int *path, int *automatic);
/* nsteps steps like gp_step on the compact split path (5) that allocate no
   memory: the cell lists live in a file-scope device array of the library (64
   MiB per GPU, held from its first use until the process ends).  No
   counterpart in the reference: this is for callers that cannot allocate --
   code under HIP graph capture, tight serving loops, harnesses that forbid
   hipMalloc.  The call only enqueues kernels on the context's stream (no
   graphs, no events, no synchronisation; gp_synchronize waits).  A grid needs
   2 + (MESH_X+2)(MESH_Y+2) + MESH_X*MESH_Y ints of the array (up to about
   2890^2 cells): larger grids return GP_E_SCRATCH.  Every call on one GPU uses
   the same array and clears its counters first; calls that overlap on one GPU
   (other streams, other threads) race.  The context's device is made current
   for the call. */
int  gp_step_noalloc(gp_ctx *ctx, long nsteps);

/* Steps run per kernel path (steps[0..6], indexed like gp_set_path) since the
   context was created or the last call with reset != 0, which clears them.
   No counterpart in the reference (it has one code path). */
int  gp_path_steps(gp_ctx *ctx, long *steps, int reset);

/* Replay gp_step calls of 32 steps or more as captured HIP graphs of 32-step
   blocks (default on).  Capture needs a non-default stream: the context owns one
   unless gp_set_stream gave another. */
int  gp_set_graphs(gp_ctx *ctx, int on);

/* Tiles of the last fused step: total, interface (full kernel) and bulk
   (diffusion-only kernel) counts; synchronises the context's stream. */
int  gp_sched_info(gp_ctx *ctx, long *ntiles, long *n_interface, long *n_bulk);

/* Tile shape of the sparse two-pass path: 0 is the default; 1..5 are further
   candidates (P <= 4): (4,64), (16,64), (8,32), (32,32), (16,32) cells. */
int  gp_set_tile_shape(gp_ctx *ctx, int shape);
/* Rows x columns of cells of the tile shape the context steps with. */
int  gp_tile_shape(gp_ctx *ctx, int *tile_x, int *tile_y);

/* Time `steps` steps of every candidate kernel path and tile shape and keep the
   fastest.  The state advances by 2 x steps per candidate; binary64 results do
   not depend on the choice. */
int  gp_autotune(gp_ctx *ctx, long steps, int *path, int *shape);

/*
 * Ensembles: n independent grids with the same P and C (sizes, constants and
 * boundaries may differ) stepped together as one tile set, so that each step of
 * the whole ensemble is one planner launch and one launch per kernel.  Blocks of
 * 32 steps are replayed as one captured HIP graph.  Member i is addressed by
 * its index; its state and statistics work as for a context.  Each member's
 * binary64 results equal those of a context of its own.
 *
 * The members share one buffer for fields in transit (gp_set_state above), as
 * large as the largest member among those within GP_TRANSIT_KEEP needs; calls on
 * different members from several threads take turns on it.
 */
typedef struct gp_ensemble gp_ensemble;
int  gp_ensemble_create(const gp_params *params, int n, int dtype, gp_ensemble **out);
void gp_ensemble_destroy(gp_ensemble *e);
int  gp_ensemble_size(gp_ensemble *e, int *n, long *cells);
int  gp_ensemble_set_state(gp_ensemble *e, int i, const double *phi, const double *mu);
int  gp_ensemble_get_state(gp_ensemble *e, int i, double *phi, double *mu);
int  gp_ensemble_step(gp_ensemble *e, long nsteps);
int  gp_ensemble_stats_get(gp_ensemble *e, int i, gp_stats *st);
int  gp_ensemble_last_step_ms(gp_ensemble *e, double *ms);
int  gp_ensemble_set_tile_shape(gp_ensemble *e, int shape);
int  gp_ensemble_autotune(gp_ensemble *e, long steps, int *tile_x, int *tile_y);
int  gp_ensemble_sched_info(gp_ensemble *e, long *ntiles, long *n_interface, long *n_bulk, int *tile_x, int *tile_y);
int  gp_ensemble_synchronize(gp_ensemble *e);

/*
 * Adjoint: gradients of L = 1/2 sum over interior cells of (phi_0(T) - target)^2
 * after T = nsteps steps of a context (two phases, one independent component,
 * BINARY), with respect to the anisotropy strength dab[0][1], the pair
 * relaxation constant Tau[0][1], the interface energy GAMMA[0][1] and the
 * liquid diffusivity, and optionally to the initial state.  The forward steps
 * run the context's two-pass kernels (the same binary64 states as every path);
 * the states are kept in nsnap snapshot slots of device memory with binomial
 * checkpointing (nsnap = 0, or nsnap >= nsteps: one slot per step holding the
 * state and its delta-phi, no recomputation).  Parameter gradients are
 * accumulated in binary64.  On return the context holds the state after the
 * last recomputed step, not necessarily the final one.
 * No reference counterpart: the serial solver has no adjoint.
 */
typedef struct gp_adjoint gp_adjoint;
int  gp_adjoint_create(gp_ctx *ctx, long nsteps, int nsnap, gp_adjoint **out);
void gp_adjoint_destroy(gp_adjoint *adj);
/* phi0/mu0: initial state (host layout above); target: P=0 plane (mesh_x*mesh_y);
   grad[4] = dL/d(dab, Tau, GAMMA, D_liquid); lam_phi0/lam_mu0 (optional): dL/d(initial state). */
int  gp_adjoint_run(gp_adjoint *adj, const double *phi0, const double *mu0, const double *target, double *loss,
                    double *grad, double *lam_phi0, double *lam_mu0);
/* device time of the forward (recomputation included) and reverse kernels of the
   last run, and the number of forward steps taken */
int  gp_adjoint_info(gp_adjoint *adj, double *fwd_ms, double *rev_ms, long *forward_steps);

/* temp_bottom of a non-isothermal run (isothermal = 0) after t steps from the
   state given to gp_set_state, with the frame moved by shift_offset rows:
   tempgrad[0] - BASE_POS*GRADIENT with
   BASE_POS = tempgrad[3]/dy - shift_offset + (tempgrad[4]/dy)*(t*dt) (the last
   term only for t > 0) and GRADIENT = tempgrad[1]*dy/tempgrad[2]; row y of the
   padded grid is at temp_bottom + y*GRADIENT.  Replaces the driver's BASE_POS /
   temp_bottom lines (microsim_gp.c:77-81, 108-113). */
double gp_temp_bottom(const gp_params *p, long shift_offset, long t);

/*
 * Moving frame in y (Shift = 1).
 * gp_check_shift: check_SHIFT of the current state (functions/shift.h:44-66,
 * folded over rows as solverloop/solverloop.h:61-66 does): the largest padded
 * y in [1, MESH_Y+5] at which the last phase goes from phi < 1/2 at y-1 to
 * phi > 1/2 at y, over the interior rows x in [3, MESH_X+2]; 0 if there is
 * none.  The reference also scans the ghost rows x = 1, 2, MESH_X+3, which
 * hold values of its sweep before the boundary copy.
 * gp_apply_shift_y: apply_shiftY (functions/shift.h:4-38) by d rows,
 * 1 <= d <= MESH_Y: every padded column, ghost layers included, moves d rows
 * towards y = 0; the top d rows become the last phase (phi = 1, the others 0)
 * at mu = mu_fill[C] (the reference's Mu(cfill of the liquid, Tfill)).  No
 * boundary copy follows, as in the reference.  For a non-isothermal run the
 * next step sees the temperature profile moved with the fields and later
 * steps use temp_bottom with the frame offset increased by d.  The next
 * gp_stats_get reports zero change; take the statistics of a step before
 * shifting, as the reference's report does.
 * No counterpart for the caller's decision (microsim_gp.c:115-126): shift by
 * pos - Shiftj when pos > Shiftj, every 100 steps.
 */
int gp_check_shift(gp_ctx *ctx, long *pos);
int gp_apply_shift_y(gp_ctx *ctx, long d, const double *mu_fill);

const char *gp_strerror(int code);

#ifdef __cplusplus
}
#endif

#endif /* GPSTEP_H_ */
