// gp_ctx.hpp -- the opaque context behind gpstep.h and the per-(P, C, real type)
// entry points that the instantiation files provide.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

#include "gpstep.h"

#define GP_GRAPH_SLOTS 6
#define GP_NPATHS 7

struct gp_ctx {
  gp_params hp;         // host copy of the parameters
  int dtype;            // GP_F64 / GP_F32
  int P, C;
  int rx, ry, pitch;
  long plane;           // elements per plane
  size_t esize;         // bytes per element
  int device;
  void *phi[2], *mu[2]; // ping-pong field buffers (padded planes)
  void *mulo[2];        // binary32 path: low-order part of mu (compensated update)
  void *dphi;           // two-pass path: delta-phi planes
  signed char *dcode;   // sparse and split two-pass paths: per-cell one-hot / zero-delta-phi code
  int *dsplit;          // split two-pass path: 2 counters, phase-sweep and mu-sweep block lists
  int *dcells;          // compact split and one-hot paths: 2 counters, phase-sweep and mu-sweep cell lists (on first use)
  int *dcells6;         // one-hot path: segmented phase-sweep and mu-sweep cell lists with their counters (on first use)
  signed char *doh;     // one-hot path: per state buffer, the exact one-hot phase of each cell or -1 (on first use)
  int oh_valid;         // doh describes both state buffers (the previous step was a one-hot path step)
  // phase-field noise (hp.noise): glibc rand() state (31 words), jump matrices,
  // the step's words, per-cell draw offsets (plane layout), per-row counts and
  // bases ([2][rx]) and the step's draw count
  unsigned int *dnz_state, *dnz_jump, *dnz_raw;
  int *dnz_off, *dnz_rows, *dnz_total;
  void *dcomp;          // composition planes (MPI semantics, GP_MPI_COMPOSITION), else null
  unsigned long long *drstate;  // drand48 state of the MPI noise, else null
  int nz_cap;
  void *dprm;           // DevParams<R> on the device
  double *dpart;        // stats partials
  int nstat_blocks;
  int cur;              // index of the current state buffers
  int stepped;          // the other buffers hold the state one step earlier
  long tstep;           // steps since the state was loaded (temperature of non-isothermal runs)
  long shift_off;       // rows the moving frame has moved since the state was loaded
  long shift_pend;      // rows of a shift not yet followed by a step (temperature of that step)
  int *drow;            // interface position per interior row (allocated on first use)
  int pow2;             // dx and dy are powers of two (binary64 steps from namespace gpk2)
  int path;             // 0 sparse fused, 1 two-pass, 2 dense fused, 3 sparse two-pass, 4 split two-pass,
                        // 5 compact split, 6 one-hot (GP_NPATHS paths)
  hipStream_t stream;
  hipEvent_t ev0, ev1;
  double last_ms;
  // sparse interface scheduling (fused path)
  int tile_tx, tile_ty;  // tile shape of the instantiated fused kernels
  int ntx, nty, ntiles, maxdep;
  int *dflag[2];         // per-tile one-hot flag of state buffers 0/1 (-1: not bulk)
  int *ddeps;            // [ntiles][maxdep+1]: count, tiles the 2-cell halo reads from
  int *dlist;            // [2][ntiles]: interface list, bulk list
  int *dlist_all;        // all tiles (dense fused path)
  int *dcnt;             // [2 step parities][interface, bulk] counters; [4],[5] = ntiles
  int cnt_par;
  int flags_valid;
  long n_if_last, n_bulk_last;
  // step graphs: GRAPH_STEPS steps captured once per starting parity
  hipStream_t own_stream;   // created with default priority when the caller sets none
  hipGraphExec_t graph[2];  // unused (see gcache)
  int graph_path;
  int use_graphs;
  // captured step blocks per (path, tile shape) and starting parity
  hipGraphExec_t gcache[GP_GRAPH_SLOTS][2];
  int gkey[GP_GRAPH_SLOTS];
  // automatic path choice: re-timed when auto_count reaches auto_next; the gap
  // starts at auto_period blocks and doubles (up to 8x) while the choice holds
  int auto_mode;
  long auto_count, auto_period, auto_next, auto_gap;
  // grids of the tile set: a context steps itself; an ensemble master (nmember
  // > 0) owns no fields and steps its member contexts as one tile set
  int nmember;
  gp_ctx **member;
  int tile0;             // first global tile of this grid in its tile set
  void *dinst;           // device Inst<R>[max(1, nmember)]
  int *dtinst;           // ensemble: global tile -> member (null for one grid)
  long path_steps[GP_NPATHS];  // steps run per kernel path since the last gp_path_steps reset
  int shape;             // tile shape of the sparse two-pass path (index into the candidate list)
  int shape_set;         // tile shape the tile set was built for (-1: none)
  // gp_set_state / gp_get_state: the context whose buffer for fields in transit
  // this one uses (itself; the master for an ensemble member), that buffer (on
  // first use), its size (0: none is kept) and the lock under which a call uses it
  gp_ctx *stage_of;
  double *stage;
  size_t stage_bytes;
  std::mutex stage_mu;
};

#define GP_GRAPH_STEPS 32

namespace gpk {

// tile shapes of the sparse two-pass path: 0 is the fused kernel's shape (the
// default), 1.. are the autotuner's further candidates (P <= 4)
constexpr int kNumShapes = 6;

// per-(P,C,R) entry points, instantiated in gp_inst_p*.hip
template <int P, int C, class R>
int run_steps(gp_ctx *c, long nsteps);
template <int P, int C, class R>
int run_steps_lists(gp_ctx *c, long nsteps, int *cells);
template <int P, int C, class R>
int run_comp_init(gp_ctx *c);
template <int P, int C, class R>
int two_pass_into(gp_ctx *c, const void *phi, const void *mu, void *dphi, const void *mulo, void *phi_o, void *mu_o,
                  void *mulo_o);
template <int P, int C, class R>
int phase_into(gp_ctx *c, const void *phi, const void *mu, void *dphi);
template <int P, int C, class R>
int run_stats(gp_ctx *c, gp_stats *st);
template <int P, int C, class R>
int run_smooth(gp_ctx *c, long nsweeps);

}  // namespace gpk

// the binary64 steps for spacings that are powers of two (gp_inst_p*.hip
// compiled with -DGP_POW2 -DGPK_NS=gpk2)
namespace gpk2 {
template <int P, int C, class R>
int run_steps(gp_ctx *c, long nsteps);
template <int P, int C, class R>
int run_steps_lists(gp_ctx *c, long nsteps, int *cells);
template <int P, int C, class R>
int run_comp_init(gp_ctx *c);
template <int P, int C, class R>
int two_pass_into(gp_ctx *c, const void *phi, const void *mu, void *dphi, const void *mulo, void *phi_o, void *mu_o,
                  void *mulo_o);
template <int P, int C, class R>
int phase_into(gp_ctx *c, const void *phi, const void *mu, void *dphi);
template <int P, int C, class R>
int run_stats(gp_ctx *c, gp_stats *st);
template <int P, int C, class R>
int run_smooth(gp_ctx *c, long nsweeps);
}  // namespace gpk2

// gp_step without the closing synchronisation when timed is false
int gp_step_impl(gp_ctx *c, long nsteps, bool timed);

#define GP_HIP_CHECK(expr)                 \
  do {                                     \
    hipError_t e_ = (expr);                \
    if (e_ != hipSuccess) return GP_E_HIP; \
  } while (0)
