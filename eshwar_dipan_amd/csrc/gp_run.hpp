// gp_run.hpp -- host-side launch sequences for one (P, C, real type); included by
// the instantiation files gp_inst_p*.hip.
#pragma once

#include <algorithm>
#include <vector>

#include "gp_ctx.hpp"
#include "gp_fused.hpp"
#include "gp_noise.hpp"

// Blocks of 256 lanes that the dense kernels of the compact split path loop
// with over their cell lists.
#ifndef GP_DENSE_BLOCKS
#define GP_DENSE_BLOCKS 2048
#endif
// Blocks of 256 lanes of the one-hot path's dense sweeps.
#ifndef GP_ONEHOT_DENSE
#define GP_ONEHOT_DENSE 512
#endif
// The one-hot path's dense phase sweep and light mu sweep as one launch (1)
// or as two (0); always two at nine or more phases.
#ifndef GP_ONEHOT_MERGED
#define GP_ONEHOT_MERGED 1
#endif

namespace GPK_NS {

// Tile of the fused kernel: the largest of (8,64), (4,64), (8,32), (4,32),
// (2,32) interior cells whose LDS staging fits in 60 KiB.
template <int P, int C, class R>
struct FusedTile {
  template <int TX, int TY>
  static constexpr bool fits = sizeof(FusedSmem<P, C, R, TX, TY>) <= 60 * 1024;
  static constexpr int TX = fits<8, 64> ? 8 : fits<4, 64> ? 4 : fits<8, 32> ? 8 : fits<4, 32> ? 4 : 2;
  static constexpr int TY = fits<8, 64> || fits<4, 64> ? 64 : 32;
};

// Tile shapes of the sparse two-pass path (TX rows x TY columns of cells).
// Shape 0 is FusedTile; the others are the autotuner's candidates for P <= 4.
template <int P, int C, class R, int S>
struct ShapeOf {
  static constexpr int TX = S == 0 ? FusedTile<P, C, R>::TX : S == 1 ? 4 : S == 2 ? 16 : S == 3 ? 8 : S == 4 ? 32 : 16;
  static constexpr int TY = S == 0 ? FusedTile<P, C, R>::TY : S == 1 ? 64 : S == 2 ? 64 : S == 3 ? 32 : S == 4 ? 32 : 32;
};
template <int P>
constexpr bool shape_allowed(int s) { return s == 0 || P <= 4; }

inline int shape_tx(int s, int tx0) { return s == 0 ? tx0 : s == 1 ? 4 : s == 2 ? 16 : s == 3 ? 8 : s == 4 ? 32 : 16; }
inline int shape_ty(int s, int ty0) { return s == 0 ? ty0 : s == 1 ? 64 : s == 2 ? 64 : s == 3 ? 32 : s == 4 ? 32 : 32; }

// Releases the tile set: the queued work that may use it finishes first, then
// the captured blocks that name its buffers go, then the buffers.
inline void free_tiles(gp_ctx *c) {
  (void)hipStreamSynchronize(c->stream);
  for (int g = 0; g < GP_GRAPH_SLOTS; g++) {
    for (int i = 0; i < 2; i++)
      if (c->gcache[g][i]) (void)hipGraphExecDestroy(c->gcache[g][i]), c->gcache[g][i] = nullptr;
    c->gkey[g] = -1;
  }
  for (int i = 0; i < 2; i++)
    if (c->dflag[i]) (void)hipFree(c->dflag[i]), c->dflag[i] = nullptr;
  if (c->ddeps) (void)hipFree(c->ddeps), c->ddeps = nullptr;
  if (c->dlist) (void)hipFree(c->dlist), c->dlist = nullptr;
  if (c->dlist_all) (void)hipFree(c->dlist_all), c->dlist_all = nullptr;
  if (c->dcnt) (void)hipFree(c->dcnt), c->dcnt = nullptr;
  if (c->dinst) (void)hipFree(c->dinst), c->dinst = nullptr;
  if (c->dtinst) (void)hipFree(c->dtinst), c->dtinst = nullptr;
  c->shape_set = -1;
}

// Ghost-aware dependency lists of one grid: tile t depends on every tile owning
// a source cell of its 2-cell halo, the halo's ghost cells mapped to their copy
// sources (bc_proxy of phi).  Indices are global (offset g->tile0).
inline void grid_deps(const gp_ctx *g, int TX, int TY, int maxdep, int *deps) {
  const long MX = g->hp.mesh_x, MY = g->hp.mesh_y;
  const int rows[2] = {g->rx, g->ry};
  auto src = [&](int axis, int v) -> int {
    long n = axis ? MY : MX;
    if (v >= 3 && v <= n + 2) return v;
    const long *lo = g->hp.bc_proxy[0][axis ? GP_FACE_YMIN : GP_FACE_XMIN];
    const long *hi = g->hp.bc_proxy[0][axis ? GP_FACE_YMAX : GP_FACE_XMAX];
    if (v <= 2) return (int)lo[2 - v];     // ghosts 2,1,0 <- proxy 0,1,2
    return (int)hi[v - (rows[axis] - 3)];  // ghosts n-3.. <- proxy 0,1,2
  };
  for (int tx = 0; tx < g->ntx; tx++)
    for (int ty = 0; ty < g->nty; ty++) {
      int sx[64], sy[128], nsx = 0, nsy = 0;
      int x0 = 3 + tx * TX, x1 = (int)std::min<long>(x0 + TX - 1, MX + 2);
      int y0 = 3 + ty * TY, y1 = (int)std::min<long>(y0 + TY - 1, MY + 2);
      for (int x = x0 - 2; x <= x1 + 2; x++) {
        int o = (src(0, x) - 3) / TX;
        bool seen = false;
        for (int i = 0; i < nsx; i++) seen |= sx[i] == o;
        if (!seen && nsx < 64) sx[nsx++] = o;
      }
      for (int y = y0 - 2; y <= y1 + 2; y++) {
        int o = (src(1, y) - 3) / TY;
        bool seen = false;
        for (int i = 0; i < nsy; i++) seen |= sy[i] == o;
        if (!seen && nsy < 128) sy[nsy++] = o;
      }
      int *d = &deps[(size_t)(g->tile0 + tx * g->nty + ty) * (maxdep + 1)];
      if (nsx * nsy > maxdep) {
        d[0] = -1;  // always an interface tile
        continue;
      }
      int n = 0;
      for (int i = 0; i < nsx; i++)
        for (int j = 0; j < nsy; j++) d[1 + n++] = g->tile0 + sx[i] * g->nty + sy[j];
      d[0] = n;
    }
}

// Tile set of a context or ensemble for tile shape TX x TY: per-grid geometry,
// dependency lists, flags, lists, counters and the device grid table.
template <class R>
int setup_tiles(gp_ctx *c, int shape, int TX, int TY) {
  if (c->dflag[0] && c->shape_set == shape) return GP_OK;
  free_tiles(c);
  const int ng = c->nmember ? c->nmember : 1;
  gp_ctx *const *grids = c->nmember ? c->member : &c;
  int total = 0;
  for (int i = 0; i < ng; i++) {
    gp_ctx *g = grids[i];
    g->tile_tx = TX;
    g->tile_ty = TY;
    g->ntx = (int)((g->hp.mesh_x + TX - 1) / TX);
    g->nty = (int)((g->hp.mesh_y + TY - 1) / TY);
    g->ntiles = g->ntx * g->nty;
    g->tile0 = total;
    total += g->ntiles;
  }
  c->tile_tx = TX;
  c->tile_ty = TY;
  c->ntiles = total;
  c->maxdep = 16;
  std::vector<int> deps((size_t)total * (c->maxdep + 1), 0);
  std::vector<int> tinst(c->nmember ? total : 0);
  std::vector<Inst<R>> inst(ng);
  for (int i = 0; i < ng; i++) {
    gp_ctx *g = grids[i];
    grid_deps(g, TX, TY, c->maxdep, deps.data());
    for (int t = 0; t < g->ntiles && c->nmember; t++) tinst[g->tile0 + t] = i;
    Inst<R> &I = inst[i];
    I.prm = (const DevParams<R> *)g->dprm;
    for (int k = 0; k < 2; k++) {
      I.phi[k] = (R *)g->phi[k];
      I.mu[k] = (R *)g->mu[k];
      I.mulo[k] = (R *)g->mulo[k];
    }
    I.dphi = (R *)g->dphi;
    I.code = g->dcode;
    I.nty = g->nty;
    I.tile0 = g->tile0;
  }
  std::vector<int> all(total);
  for (int i = 0; i < total; i++) all[i] = i;
  size_t nt = (size_t)total;
  GP_HIP_CHECK(hipMalloc((void **)&c->dflag[0], nt * sizeof(int)));
  GP_HIP_CHECK(hipMalloc((void **)&c->dflag[1], nt * sizeof(int)));
  GP_HIP_CHECK(hipMalloc((void **)&c->ddeps, deps.size() * sizeof(int)));
  GP_HIP_CHECK(hipMalloc((void **)&c->dlist, 2 * nt * sizeof(int)));
  GP_HIP_CHECK(hipMalloc((void **)&c->dlist_all, nt * sizeof(int)));
  GP_HIP_CHECK(hipMalloc((void **)&c->dcnt, 8 * sizeof(int)));
  GP_HIP_CHECK(hipMalloc(&c->dinst, ng * sizeof(Inst<R>)));
  if (c->nmember) GP_HIP_CHECK(hipMalloc((void **)&c->dtinst, nt * sizeof(int)));
  int cnt0[8] = {0, 0, 0, 0, total, total, 0, 0};
  GP_HIP_CHECK(hipMemcpy(c->ddeps, deps.data(), deps.size() * sizeof(int), hipMemcpyHostToDevice));
  GP_HIP_CHECK(hipMemcpy(c->dlist_all, all.data(), nt * sizeof(int), hipMemcpyHostToDevice));
  GP_HIP_CHECK(hipMemcpy(c->dcnt, cnt0, sizeof(cnt0), hipMemcpyHostToDevice));
  GP_HIP_CHECK(hipMemcpy(c->dinst, inst.data(), ng * sizeof(Inst<R>), hipMemcpyHostToDevice));
  if (c->nmember) GP_HIP_CHECK(hipMemcpy(c->dtinst, tinst.data(), nt * sizeof(int), hipMemcpyHostToDevice));
  // these copies run on the null stream, which the context's non-blocking
  // stream does not wait for: they land before the kernels that read them
  GP_HIP_CHECK(hipStreamSynchronize(nullptr));
  c->cnt_par = 0;
  c->flags_valid = 0;
  c->shape_set = shape;
  return GP_OK;
}

// Sparse steps (paths 0, 2, 3) with tile shape S.
template <int P, int C, class R, int S>
int run_sparse(gp_ctx *c, long nsteps) {
  using T = ShapeOf<P, C, R, S>;
  int rc = setup_tiles<R>(c, S, T::TX, T::TY);
  if (rc) return rc;
  const int nt = c->ntiles;
  const Inst<R> *inst = (const Inst<R> *)c->dinst;
  const int *tinst = c->dtinst;
  // The counter pair of a step is chosen by cnt_par, the state buffers by cur.
  // Anything else that steps the state (two-pass and split steps, smoothing,
  // frame shifts, the adjoint) flips cur alone and clears flags_valid; so with
  // fresh flags both counter pairs are cleared and the pairs are tied to the
  // state parity again.  Captured sparse blocks (cached by cur) then always
  // meet the counter pair they were captured with.
  if (!c->flags_valid || c->cnt_par != c->cur) {
    hipLaunchKernelGGL(k_clear_counts<0>, dim3(1), dim3(64), 0, c->stream, c->dcnt);
    c->cnt_par = c->cur;
    hipLaunchKernelGGL((k_flags<P, R, T::TX, T::TY>), dim3(nt), dim3(256), 0, c->stream, inst, tinst, c->cur,
                       c->dflag[c->cur], c->dflag[c->cur ^ 1]);
    c->flags_valid = 1;
  }
  const int g_if = std::min(nt, 2048), g_bulk = std::min(nt, 4096);
  for (long t = 0; t < nsteps; t++) {
    int i = c->cur, o = c->cur ^ 1;
    int *cnt = c->dcnt + 2 * c->cnt_par, *cnt_next = c->dcnt + 2 * (c->cnt_par ^ 1);
    const int *list_if = c->dlist, *cnt_if = cnt;
    if (c->path != 2) {
      hipLaunchKernelGGL(k_plan<0>, dim3((nt + 255) / 256), dim3(256), 0, c->stream, (const int *)c->dflag[i],
                         (const int *)c->ddeps, c->maxdep, nt, c->dlist, c->dlist + nt, cnt, cnt_next);
    } else {
      list_if = c->dlist_all;
      cnt_if = c->dcnt + 4;
    }
    if (c->path == 3) {
      hipLaunchKernelGGL((k_phase_tiles<P, C, R, T::TX, T::TY>), dim3(g_if), dim3(256), 0, c->stream, inst, tinst, i,
                         list_if, cnt_if, nt);
      hipLaunchKernelGGL((k_conc_tiles<P, C, R, T::TX, T::TY>), dim3(g_if), dim3(256), 0, c->stream, inst, tinst, i,
                         list_if, cnt_if, c->dflag[o], nt);
    } else if constexpr (S == 0) {
      const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
      hipLaunchKernelGGL((k_fused<P, C, R, T::TX, T::TY>), dim3(g_if), dim3(256), 0, c->stream, prm,
                         (const R *)c->phi[i], (const R *)c->mu[i], (const R *)c->mulo[i], (R *)c->phi[o],
                         (R *)c->mu[o], (R *)c->mulo[o], list_if, cnt_if, c->dflag[o], c->nty, nt);
    }
    if (c->path != 2)
      hipLaunchKernelGGL((k_bulk<P, C, R, T::TX, T::TY>), dim3(g_bulk), dim3(256), 0, c->stream, inst, tinst, i,
                         (const int *)(c->dlist + nt), (const int *)(cnt + 1), (const int *)c->dflag[i], c->dflag[o],
                         nt);
    c->cur = o;
    c->cnt_par ^= 1;
  }
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// temp_bottom after t steps of a non-isothermal run whose frame has moved by
// shift_off rows, in binary64 as the reference forms it (microsim_gp.c:78-80,
// 109-111)
inline double temp_bottom(const gp_params &h, long shift_off, long t) { return gp_temp_bottom(&h, shift_off, t); }

// Phase-field noise of the coming phase sweep of `phi` (a context with
// hp.noise): counts and offsets of the draws, the step's words, and the
// generator state after them.  Kernels only, so a captured block replays the
// sequence onward.
template <int P, class R>
NoiseRef noise_prep(gp_ctx *c, const R *phi) {
  if (!c->dnz_raw) return NoiseRef{};
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  int *rcnt = c->dnz_rows, *rbase = c->dnz_rows + c->rx;
  hipLaunchKernelGGL((k_noise_count<P, R>), dim3(c->rx - 2), dim3(256), 0, c->stream, prm, phi, c->dnz_off, rcnt);
  hipLaunchKernelGGL(k_noise_scan<0>, dim3(1), dim3(1024), 0, c->stream, (const int *)rcnt, rbase, c->rx, c->dnz_total);
  const int nchunk = (c->nz_cap + NZ_CHUNK - 1) / NZ_CHUNK;
  hipLaunchKernelGGL(k_noise_gen<0>, dim3(std::max(1, std::min((nchunk + 63) / 64, 1024))), dim3(64), 0, c->stream,
                     (const uint32_t *)c->dnz_state, (const uint32_t *)c->dnz_jump, (const int *)c->dnz_total,
                     c->nz_cap, (uint32_t *)c->dnz_raw);
  hipLaunchKernelGGL(k_noise_adv<0>, dim3(1), dim3(32), 0, c->stream, (uint32_t *)c->dnz_state,
                     (const uint32_t *)c->dnz_raw, (const int *)c->dnz_total, c->nz_cap);
  return NoiseRef{(const uint32_t *)c->dnz_raw, c->dnz_off, rbase, c->hp.amp_noise};
}

// Split two-pass steps (path 4): per sweep a light kernel over the grid that
// finishes the cells with an exact shortcut and lists the blocks that hold
// others, then the dense kernel over the listed blocks only.  The dense
// kernels take a 1-D grid of every block; blocks past the list's count return
// at once.  Non-isothermal steps take the temperature arguments of run_steps.
template <int P, int C, class R, bool NI>
int run_split(gp_ctx *c, long nsteps) {
  static_assert(KM == 1, "the split mu sweep assumes one row per wave");
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  const dim3 blk(BX, BY);
  const dim3 gp = phase_grid(c->rx, c->ry);
  const dim3 gc(((int)c->hp.mesh_y + MW - 1) / MW, ((int)c->hp.mesh_x + BY - 1) / BY);
  int *cnt = c->dsplit, *lp = cnt + 2, *lc = lp + gp.x * gp.y;
  const signed char *code = (const signed char *)c->dcode;
  for (long t = 0; t < nsteps; t++) {
    const R *phi = (const R *)c->phi[c->cur], *mu = (const R *)c->mu[c->cur], *mulo = (const R *)c->mulo[c->cur];
    R *phi_o = (R *)c->phi[c->cur ^ 1], *mu_o = (R *)c->mu[c->cur ^ 1], *mulo_o = (R *)c->mulo[c->cur ^ 1];
    R *dphi = (R *)c->dphi;
    R tb = R(0);
    int tmode = 0, tsh = 0;
    if constexpr (NI) {  // as in run_steps
      const long k = c->tstep + t;
      tsh = t == 0 ? (int)c->shift_pend : 0;
      tb = (R)temp_bottom(c->hp, c->shift_off - tsh, k);
      tmode = (k == 0 ? 1 : 0) | (tsh << 1);
    }
    const NoiseRef nz = noise_prep<P, R>(c, phi);
    hipLaunchKernelGGL((k_phase_split<P, R>), gp, blk, 0, c->stream, prm, phi, dphi, c->dcode, lp, cnt);
    hipLaunchKernelGGL((k_phase<P, C, R, NI>), dim3(gp.x * gp.y), blk, 0, c->stream, prm, phi, mu, dphi, tb, tmode,
                       (const int *)lp, (const int *)cnt, (int)gp.x, nz);
    hipLaunchKernelGGL((k_conc_split<P, C, R, NI>), gc, blk, 0, c->stream, prm, phi, mu, mulo, code, phi_o, mu_o,
                       mulo_o, lc, cnt, tb, tsh);
    if constexpr (Ops<R>::Exact)
      hipLaunchKernelGGL((k_conc_lds<P, C, R, NI>), dim3(gc.x * gc.y), blk, 0, c->stream, prm, phi, mu, (const R *)dphi,
                         mulo, phi_o, mu_o, mulo_o, tb, tsh, (const int *)lc, (const int *)(cnt + 1), (int)gc.x, code);
    else
      hipLaunchKernelGGL((k_conc_march<P, C, R, NI>), dim3(gc.x * gc.y), blk, 0, c->stream, prm, phi, mu,
                         (const R *)dphi, mulo, phi_o, mu_o, mulo_o, tb, tsh, (const int *)lc, (const int *)(cnt + 1),
                         (int)gc.x, code);
    c->cur ^= 1;
  }
  if (nsteps > 0) c->shift_pend = 0;
  c->flags_valid = 0;
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// Compact split steps (path 5): per sweep a light kernel over the grid that
// finishes the cells with an exact shortcut and lists every other cell, then
// the dense kernel over the listed cells, one per lane.  The dense kernels
// loop over their list from a fixed grid.
// Cell-list buffer of the compact split path: 2 counters, the phase-sweep
// list and the mu-sweep list (ints).
inline size_t compact_list_ints(const gp_ctx *c) {
  return 2 + (size_t)(c->rx - 4) * (c->ry - 4) + (size_t)c->hp.mesh_x * c->hp.mesh_y;
}

// Steps of the compact split path with the cell lists in `cells`
// (compact_list_ints ints; counters zero, or left by a previous step).
template <int P, int C, class R, bool NI>
int run_compact_in(gp_ctx *c, long nsteps, int *cells) {
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  const dim3 blk(BX, BY);
  const dim3 gp = phase_grid(c->rx, c->ry);
  const dim3 gl(((int)c->hp.mesh_y + BX - 1) / BX, ((int)c->hp.mesh_x + BY - 1) / BY);
  const int capp = (c->rx - 4) * (c->ry - 4), capc = (int)(c->hp.mesh_x * c->hp.mesh_y);
  int *cnt = cells, *lp = cnt + 2, *lc = lp + capp;
  const signed char *code = (const signed char *)c->dcode;
  const int gdense = std::max(1, std::min((capp + 255) / 256, GP_DENSE_BLOCKS));
  for (long t = 0; t < nsteps; t++) {
    const R *phi = (const R *)c->phi[c->cur], *mu = (const R *)c->mu[c->cur], *mulo = (const R *)c->mulo[c->cur];
    R *phi_o = (R *)c->phi[c->cur ^ 1], *mu_o = (R *)c->mu[c->cur ^ 1], *mulo_o = (R *)c->mulo[c->cur ^ 1];
    R *dphi = (R *)c->dphi;
    R tb = R(0);
    int tmode = 0, tsh = 0;
    if constexpr (NI) {  // as in run_steps
      const long k = c->tstep + t;
      tsh = t == 0 ? (int)c->shift_pend : 0;
      tb = (R)temp_bottom(c->hp, c->shift_off - tsh, k);
      tmode = (k == 0 ? 1 : 0) | (tsh << 1);
    }
    const NoiseRef nz = noise_prep<P, R>(c, phi);
    hipLaunchKernelGGL((k_phase_light<P, R>), gp, blk, 0, c->stream, prm, phi, dphi, c->dcode, lp, cnt, capp);
    hipLaunchKernelGGL((k_phase_cells<P, C, R, NI>), dim3(gdense), dim3(256), 0, c->stream, prm, phi, mu, dphi, tb,
                       tmode, (const int *)lp, (const int *)cnt, capp, nz);
    hipLaunchKernelGGL((k_conc_light<P, C, R, NI>), gl, blk, 0, c->stream, prm, phi, mu, mulo, code, phi_o, mu_o,
                       mulo_o, lc, cnt, capc, tb, tsh);
    hipLaunchKernelGGL((k_conc_cells<P, C, R, NI>), dim3(gdense), dim3(256), 0, c->stream, prm, phi, mu,
                       (const R *)dphi, mulo, phi_o, mu_o, mulo_o, tb, tsh, (const int *)lc, cnt, capc, code);
    c->cur ^= 1;
  }
  if (nsteps > 0) c->shift_pend = 0;
  c->flags_valid = 0;
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// The context's cell lists of the compact split path (on first use).
inline int ensure_cells(gp_ctx *c) {
  if (!c->dcells) {
    if (c->rx > 65535 || c->ry > 65535) return GP_E_UNSUPPORTED;  // list entries pack x and y in 16 bits
    GP_HIP_CHECK(hipMalloc((void **)&c->dcells, sizeof(int) * compact_list_ints(c)));
    // the counters start at zero: cleared on the context's stream, so the
    // clear is ordered before the step kernels (a plain hipMemset runs on the
    // null stream, which a non-blocking stream does not wait for)
    hipLaunchKernelGGL(k_clear_counts<0>, dim3(1), dim3(64), 0, c->stream, c->dcells);
  }
  return GP_OK;
}

template <int P, int C, class R, bool NI>
int run_compact(gp_ctx *c, long nsteps) {
  if (int rc = ensure_cells(c)) return rc;
  return run_compact_in<P, C, R, NI>(c, nsteps, c->dcells);
}

// Steps of the one-hot path (6): per step k_phase_light_oh, k_phase_conc_oh
// (the dense phase sweep on its first nd blocks, the light mu sweep on the
// rest) and k_conc_cells_oh with the one-hot plane of the output buffer.  The
// planes (c->doh, one per state buffer) are set up from the current buffer
// when the previous step was not a step of this path (c->oh_valid == 0), also
// for nsteps == 0, so that a graph captured after such a call starts valid.
// The segmented lists and their counters live in c->dcells6 (kSegInts
// counters, then a slot for every cell of each light launch's blocks:
// kPhaseCells per block of the phase sweep, kMuCells per block of the mu sweep).
template <int P, int C, class R, bool NI>
int run_onehot(gp_ctx *c, long nsteps) {
  if (c->rx > 65535 || c->ry > 65535) return GP_E_UNSUPPORTED;  // list entries pack x and y in 16 bits
  const dim3 blk(BX, BY);
  const dim3 gp = phase_light_grid(c->rx, c->ry);
  const int gx = ((int)c->hp.mesh_y + BX - 1) / BX, gy = ((int)c->hp.mesh_x + BY - 1) / BY;
  const int nbp = (int)(gp.x * gp.y), nbc = gx * gy, capp = nbp * kPhaseCells;
  if (!c->dcells6) {
    GP_HIP_CHECK(hipMalloc((void **)&c->dcells6, sizeof(int) * ((size_t)kSegInts + (size_t)capp + (size_t)nbc * kMuCells)));
    hipLaunchKernelGGL(k_clear_seg<0>, dim3(1), dim3(256), 0, c->stream, c->dcells6);
  }
  if (!c->doh) {
    GP_HIP_CHECK(hipMalloc((void **)&c->doh, 2 * (size_t)c->plane));
    c->oh_valid = 0;
  }
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  signed char *oh[2] = {c->doh, c->doh + c->plane};
  if (!c->oh_valid) {
    hipLaunchKernelGGL((k_oh_prime<P, R>), dim3(gx, gy), blk, 0, c->stream, prm, (const R *)c->phi[c->cur],
                       oh[c->cur], oh[c->cur ^ 1]);
    c->oh_valid = 1;
  }
  // dense blocks of the merged launch (a multiple of 8, so that the light
  // blocks keep the hardware's round-robin over the 8 XCDs) and of k_conc_cells_oh
  const int nd = std::min((nbp * kPhaseCols + 7) / 8 * 8, GP_ONEHOT_DENSE);
  const int gdense = std::min(nbc, GP_ONEHOT_DENSE);
  for (long t = 0; t < nsteps; t++) {
    const R *phi = (const R *)c->phi[c->cur], *mu = (const R *)c->mu[c->cur], *mulo = (const R *)c->mulo[c->cur];
    R *phi_o = (R *)c->phi[c->cur ^ 1], *mu_o = (R *)c->mu[c->cur ^ 1], *mulo_o = (R *)c->mulo[c->cur ^ 1];
    R *dphi = (R *)c->dphi;
    R tb = R(0);
    int tmode = 0, tsh = 0;
    if constexpr (NI) {  // as in run_steps
      const long k = c->tstep + t;
      tsh = t == 0 ? (int)c->shift_pend : 0;
      tb = (R)temp_bottom(c->hp, c->shift_off - tsh, k);
      tmode = (k == 0 ? 1 : 0) | (tsh << 1);
    }
    const NoiseRef nz = noise_prep<P, R>(c, phi);
    hipLaunchKernelGGL((k_phase_light_oh<P, R>), gp, blk, 0, c->stream, prm, phi, (const signed char *)oh[c->cur],
                       dphi, c->dcode, c->dcells6);
    if constexpr (GP_ONEHOT_MERGED && !onehot_wide<P, R>()) {
      hipLaunchKernelGGL((k_phase_conc_oh<P, C, R, NI>), dim3(nd + nbc), blk, 0, c->stream, prm, phi, mu, mulo, dphi,
                         (const signed char *)c->dcode, phi_o, mu_o, mulo_o, oh[c->cur ^ 1], c->dcells6, nbp, capp,
                         nd, gx, tb, tmode, tsh, nz);
    } else {
      hipLaunchKernelGGL((k_phase_cells_oh<P, C, R, NI>), dim3(nd), dim3(256), 0, c->stream, prm, phi, mu, dphi,
                         (const int *)c->dcells6, nbp, tb, tmode, nz);
      hipLaunchKernelGGL((k_conc_light_oh<P, C, R, NI>), dim3(gx, gy), blk, 0, c->stream, prm, mu, mulo,
                         (const signed char *)c->dcode, phi_o, mu_o, mulo_o, oh[c->cur ^ 1], c->dcells6, capp, tb,
                         tsh);
    }
    hipLaunchKernelGGL((k_conc_cells_oh<P, C, R, NI>), dim3(gdense), dim3(256), 0, c->stream, prm, phi, mu,
                       (const R *)dphi, mulo, phi_o, mu_o, mulo_o, tb, tsh, c->dcells6, capp, nbc,
                       (const signed char *)c->dcode, oh[c->cur ^ 1]);
    c->cur ^= 1;
  }
  if (nsteps > 0) c->shift_pend = 0;
  c->flags_valid = 0;
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// Compact split steps with the cell lists in a caller-provided device buffer
// of at least compact_list_ints ints; the counters are cleared first.
// Launches kernels only: no allocation, no synchronisation.
template <int P, int C, class R>
int run_steps_lists(gp_ctx *c, long nsteps, int *cells) {
  if (c->rx > 65535 || c->ry > 65535) return GP_E_UNSUPPORTED;
  c->oh_valid = 0;
  hipLaunchKernelGGL(k_clear_counts<0>, dim3(1), dim3(64), 0, c->stream, cells);
  const int rc = c->hp.isothermal ? run_compact_in<P, C, R, false>(c, nsteps, cells)
                                  : run_compact_in<P, C, R, true>(c, nsteps, cells);
  if (!rc && nsteps > 0) c->path_steps[5] += nsteps;
  return rc;
}

// Steps with the MPI solver's semantics (gp_params.mpi): k_phase_mpi, the
// drand48 state advance when noise is drawn, k_conc_mpi.  Binary64 and
// isothermal contexts only (checked at creation).
template <int P, int C, class R>
int run_mpi(gp_ctx *c, long nsteps) {
  if constexpr (!Ops<R>::Exact) {
    return GP_E_UNSUPPORTED;
  } else {
    const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
    const dim3 blk(BX, BY);
    const dim3 gp = phase_grid(c->rx, c->ry);
    const dim3 gc(((int)c->hp.mesh_y + BX - 1) / BX, ((int)c->hp.mesh_x + BY - 1) / BY);
    const bool draws = (c->hp.mpi & GP_MPI_NOISE) && c->hp.noise;
    for (long t = 0; t < nsteps; t++) {
      const R *phi = (const R *)c->phi[c->cur], *mu = (const R *)c->mu[c->cur];
      hipLaunchKernelGGL((k_phase_mpi<P, C, R>), gp, blk, 0, c->stream, prm, phi, mu, (R *)c->dphi);
      if (draws) hipLaunchKernelGGL((k_lcg_advance<R>), dim3(1), dim3(64), 0, c->stream, prm);
      hipLaunchKernelGGL((k_conc_mpi<P, C, R>), gc, blk, 0, c->stream, prm, phi, mu, (const R *)c->dphi,
                         (R *)c->phi[c->cur ^ 1], (R *)c->mu[c->cur ^ 1]);
      c->cur ^= 1;
    }
    if (nsteps > 0) c->shift_pend = 0;
    c->flags_valid = 0;
    GP_HIP_CHECK(hipGetLastError());
    return GP_OK;
  }
}

// Composition planes from the current fields (k_comp_init).
template <int P, int C, class R>
int run_comp_init(gp_ctx *c) {
  if (!c->dcomp) return GP_E_UNSUPPORTED;
  const dim3 g(((int)c->hp.mesh_y + 255) / 256, (unsigned)c->hp.mesh_x);
  hipLaunchKernelGGL((k_comp_init<P, C, R>), g, dim3(256), 0, c->stream, (const DevParams<R> *)c->dprm,
                     (const R *)c->phi[c->cur], (const R *)c->mu[c->cur]);
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// One two-pass step between caller buffers (padded planes of the context's
// layout): delta-phi into dphi, the new state into phi_o / mu_o / mulo_o.
// The adjoint's forward steps use it to step its snapshot slots.
template <int P, int C, class R>
int two_pass_into(gp_ctx *c, const void *phi, const void *mu, void *dphi, const void *mulo, void *phi_o, void *mu_o,
                  void *mulo_o) {
  launch_two_pass<P, C, R>((const DevParams<R> *)c->dprm, c->rx, c->ry, (int)c->hp.mesh_x, (int)c->hp.mesh_y,
                           c->stream, (const R *)phi, (const R *)mu, (R *)dphi, (const R *)mulo, (R *)phi_o,
                           (R *)mu_o, (R *)mulo_o);
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// The phase sweep alone between caller buffers: delta-phi of (phi, mu) into
// dphi.  The adjoint recomputes delta-phi of a recomputed state with it.
template <int P, int C, class R>
int phase_into(gp_ctx *c, const void *phi, const void *mu, void *dphi) {
  hipLaunchKernelGGL((k_phase<P, C, R>), phase_grid(c->rx, c->ry), dim3(BX, BY), 0, c->stream,
                     (const DevParams<R> *)c->dprm, (const R *)phi, (const R *)mu, (R *)dphi, R(0), 0,
                     (const int *)nullptr, (const int *)nullptr, 0, NoiseRef{});
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

template <int P, int C, class R>
int run_steps(gp_ctx *c, long nsteps) {
  if (c->path != 6 || c->hp.mpi) c->oh_valid = 0;  // the one-hot planes hold only across the one-hot path's steps
  if (c->hp.mpi) return run_mpi<P, C, R>(c, nsteps);
  if (c->path == 6) return c->hp.isothermal ? run_onehot<P, C, R, false>(c, nsteps) : run_onehot<P, C, R, true>(c, nsteps);
  if (c->path == 5) return c->hp.isothermal ? run_compact<P, C, R, false>(c, nsteps) : run_compact<P, C, R, true>(c, nsteps);
  if (c->path == 4) return c->hp.isothermal ? run_split<P, C, R, false>(c, nsteps) : run_split<P, C, R, true>(c, nsteps);
  if (c->path == 0 || c->path == 2 || c->path == 3) {
    if (c->hp.noise) return GP_E_UNSUPPORTED;  // the tile engines draw no noise
    // the fused kernel (paths 0, 2) and ensembles of grids use their own constraints
    int s = (c->path == 3 && shape_allowed<P>(c->shape)) ? c->shape : 0;
    switch (s) {
      case 1: if constexpr (shape_allowed<P>(1)) return run_sparse<P, C, R, 1>(c, nsteps); break;
      case 2: if constexpr (shape_allowed<P>(2)) return run_sparse<P, C, R, 2>(c, nsteps); break;
      case 3: if constexpr (shape_allowed<P>(3)) return run_sparse<P, C, R, 3>(c, nsteps); break;
      case 4: if constexpr (shape_allowed<P>(4)) return run_sparse<P, C, R, 4>(c, nsteps); break;
      case 5: if constexpr (shape_allowed<P>(5)) return run_sparse<P, C, R, 5>(c, nsteps); break;
      default: break;
    }
    return run_sparse<P, C, R, 0>(c, nsteps);
  }
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  for (long t = 0; t < nsteps; t++) {
    const NoiseRef nz = noise_prep<P, R>(c, (const R *)c->phi[c->cur]);
    if (c->hp.isothermal) {
      launch_two_pass<P, C, R>(prm, c->rx, c->ry, (int)c->hp.mesh_x, (int)c->hp.mesh_y, c->stream,
                               (const R *)c->phi[c->cur], (const R *)c->mu[c->cur], (R *)c->dphi,
                               (const R *)c->mulo[c->cur], (R *)c->phi[c->cur ^ 1], (R *)c->mu[c->cur ^ 1],
                               (R *)c->mulo[c->cur ^ 1], R(0), 0, 0, nz);
    } else {
      // step k = tstep + t + 1 sees the temperature set after step k-1; its phase
      // sweep sees the temperature boundary copies only in the first step.  A
      // step right after a shift of the frame sees that profile moved with the
      // fields, in the frame before the shift.
      const long k = c->tstep + t;
      const long tsh = t == 0 ? c->shift_pend : 0;
      launch_two_pass<P, C, R, true>(prm, c->rx, c->ry, (int)c->hp.mesh_x, (int)c->hp.mesh_y, c->stream,
                                     (const R *)c->phi[c->cur], (const R *)c->mu[c->cur], (R *)c->dphi,
                                     (const R *)c->mulo[c->cur], (R *)c->phi[c->cur ^ 1], (R *)c->mu[c->cur ^ 1],
                                     (R *)c->mulo[c->cur ^ 1], (R)temp_bottom(c->hp, c->shift_off - tsh, k),
                                     k == 0 ? 1 : 0, (int)tsh, nz);
    }
    c->cur ^= 1;
  }
  if (nsteps > 0) c->shift_pend = 0;
  c->flags_valid = 0;
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

template <int P, int C, class R>
int run_smooth(gp_ctx *c, long nsweeps) {
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  dim3 blk(BX, BY);
  dim3 g((c->hp.mesh_y + BX - 1) / BX, (c->hp.mesh_x + BY - 1) / BY);
  for (long t = 0; t < nsweeps; t++) {
    hipLaunchKernelGGL((k_smooth<P, C, R>), g, blk, 0, c->stream, prm, (const R *)c->phi[c->cur],
                       (const R *)c->mu[c->cur], (const R *)c->mulo[c->cur], (R *)c->phi[c->cur ^ 1],
                       (R *)c->mu[c->cur ^ 1], (R *)c->mulo[c->cur ^ 1]);
    c->cur ^= 1;
  }
  c->flags_valid = 0;
  c->oh_valid = 0;
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

template <int P, int C, class R>
int run_stats(gp_ctx *c, gp_stats *st) {
  constexpr int NE = 3 * P + 3 * C + 1 + P + C, NV = NE + 4;
  const DevParams<R> *prm = (const DevParams<R> *)c->dprm;
  const R *pp = c->stepped ? (const R *)c->phi[c->cur ^ 1] : nullptr;
  const R *mp = c->stepped ? (const R *)c->mu[c->cur ^ 1] : nullptr;
  hipLaunchKernelGGL((k_stats<P, C, R>), dim3(c->nstat_blocks), dim3(256), 0, c->stream, prm,
                     (const R *)c->phi[c->cur], (const R *)c->mu[c->cur], pp, mp, c->dpart,
                     c->hp.isothermal ? 0.0 : temp_bottom(c->hp, c->shift_off, c->tstep));
  GP_HIP_CHECK(hipGetLastError());
  std::vector<double> h((size_t)c->nstat_blocks * NV);
  GP_HIP_CHECK(hipMemcpyAsync(h.data(), c->dpart, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  for (int a = 0; a < P; a++) { st->phi_max[a] = -INFINITY; st->phi_min[a] = INFINITY; st->phi_sum[a] = 0; }
  for (int k = 0; k < C; k++) { st->mu_max[k] = -INFINITY; st->mu_min[k] = INFINITY; st->solute[k] = 0; }
  st->nonfinite = 0;
  for (int b = 0; b < c->nstat_blocks; b++) {
    const double *v = &h[(size_t)b * NV];
    for (int a = 0; a < P; a++) {
      st->phi_max[a] = fmax(st->phi_max[a], v[a]);
      st->phi_min[a] = fmin(st->phi_min[a], v[P + a]);
      st->phi_sum[a] += v[2 * P + a];
    }
    for (int k = 0; k < C; k++) {
      st->mu_max[k] = fmax(st->mu_max[k], v[3 * P + k]);
      st->mu_min[k] = fmin(st->mu_min[k], v[3 * P + C + k]);
      st->solute[k] += v[3 * P + 2 * C + k];
    }
    st->nonfinite += v[3 * P + 3 * C];
    for (int a = 0; a < P; a++) st->rel_change_phi[a] += v[3 * P + 3 * C + 1 + a];
    for (int k = 0; k < C; k++) st->rel_change_mu[k] += v[3 * P + 3 * C + 1 + P + k];
    st->energy_gradient += v[NE];
    st->energy_potential += v[NE + 1];
    st->energy_bulk += v[NE + 2];
    st->free_energy += v[NE + 3];  // sum mu.c for now
  }
  st->grand_potential = st->energy_gradient + st->energy_potential + st->energy_bulk;
  st->free_energy += st->grand_potential;
  return GP_OK;
}

}  // namespace GPK_NS

#define GP_INSTANTIATE(P, C, R)                                \
  template int GPK_NS::run_steps<P, C, R>(gp_ctx *, long);    \
  template int GPK_NS::run_steps_lists<P, C, R>(gp_ctx *, long, int *); \
  template int GPK_NS::run_comp_init<P, C, R>(gp_ctx *);       \
  template int GPK_NS::two_pass_into<P, C, R>(gp_ctx *, const void *, const void *, void *, const void *, void *, \
                                              void *, void *);                                                  \
  template int GPK_NS::phase_into<P, C, R>(gp_ctx *, const void *, const void *, void *); \
  template int GPK_NS::run_smooth<P, C, R>(gp_ctx *, long);   \
  template int GPK_NS::run_stats<P, C, R>(gp_ctx *, gp_stats *);
