// gp_fused.hpp -- one-launch step: LDS-staged tile of TX x TY interior cells.
//
//   1. phi of the tile plus a 2-cell halo and mu plus a 1-cell halo are read
//      from HBM once into LDS (every field value of the step is read once per
//      tile; halo re-reads hit L2);
//   2. delta-phi is computed for the tile plus a 1-cell ring into LDS (the ring
//      is the neighbours' delta-phi that the antitrapping flux needs);
//   3. mu and phi of the tile are updated and written once, together with the
//      ghost cells that copy them.
// The arithmetic per value is the cell/face functions of gp_cell.hpp, so the
// binary64 instantiation equals the two-pass kernels bit for bit.
//
// binary32: mu carries a low-order word (mulo); the interface and bulk mu
// increments are added with Kahan compensation, and the bulk update is applied as
// the increment dMu/dc . delta_c of the linear F_01 map instead of Mu(c(mu)+dc),
// which is the same value in exact arithmetic without the round trip through c.
#pragma once

#include "gp_kernels.hpp"

namespace GPK_NS {

template <int P, int C, class R, int TX, int TY>
struct FusedSmem {
  static constexpr int RX2 = TX + 4, RY2 = TY + 4;  // phi region (halo 2)
  static constexpr int RX1 = TX + 2, RY1 = TY + 2;  // mu / delta-phi region (halo 1)
  R phi[P][RX2][RY2];
  R mu[C][RX1][RY1];
  R dp[P][RX1][RY1];
};

// One grid of a tile set: its parameters, ping-pong fields and scratch planes,
// its tile-row count and the global index of its first tile.  A context is a
// set of one grid; an ensemble concatenates the tiles of all its grids, and
// every tile-list kernel looks its grid up per tile (tinst: global tile ->
// grid; null when there is one grid).
template <class R>
struct Inst {
  const DevParams<R>* prm;
  R* phi[2];
  R* mu[2];
  R* mulo[2];
  R* dphi;
  signed char* code;
  int nty;
  int tile0;
};

template <class R>
__device__ __forceinline__ const Inst<R>& inst_of(const Inst<R>* __restrict__ inst, const int* __restrict__ tinst,
                                                  int tile) {
  return inst[tinst ? tinst[tile] : 0];
}

// One-hot code of a cell on the split paths (4, 5): the phase a if phi is one-hot
// in a (phi_a == 1, all others == 0 of either sign), -1 otherwise.
template <int P, class R>
__device__ __forceinline__ int onehot_phase(const R* ph) {
  int a1 = -1, nz = 0;
#pragma unroll
  for (int a = 0; a < P; a++) {
    if (ph[a] == R(1.0)) a1 = a;
    else if (ph[a] != R(0)) nz++;
  }
  return nz == 0 ? a1 : -1;
}

// Exact one-hot code of a phase vector (tile flags, the tile paths' cell codes and
// the one-hot path): a if ph is bit for bit the one-hot vector of phase a (1 in a,
// +0 in every other phase), -1 otherwise.
template <int P, class R>
__device__ __forceinline__ int onehot_bits(const R* ph) {
  int a1 = -1, n1 = 0;
  bool z = true;
#pragma unroll
  for (int a = 0; a < P; a++) {
    if (ph[a] == R(1.0)) {
      a1 = a;
      n1++;
    } else {
      z = z && ph[a] == R(0) && !signbit(ph[a]);
    }
  }
  return z && n1 == 1 ? a1 : -1;
}

// Tile flags: one phase for all cells, or -1; -2 marks "no cell" in reductions.
__device__ __forceinline__ int flag_combine(int x, int y) { return x == -2 ? y : y == -2 ? x : (x == y ? x : -1); }

// Block-wide combination of per-thread flags; result valid in thread 0.
__device__ __forceinline__ int block_flag(int f, int* red) {
  red[threadIdx.x] = f;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = flag_combine(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  int r = red[0];
  __syncthreads();
  return r;
}

template <int P, int C, class R, int TX, int TY>
__global__ void __launch_bounds__(256) GP_HEAVY k_fused(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                               const R* __restrict__ mu, const R* __restrict__ mulo,
                                               R* __restrict__ phi_o, R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                               const int* __restrict__ list, const int* __restrict__ count,
                                               int* __restrict__ flag_o, int nty, int cap) {
  using S = FusedSmem<P, C, R, TX, TY>;
  constexpr int RX2 = S::RX2, RY2 = S::RY2, RX1 = S::RX1, RY1 = S::RY1;
  __shared__ S sm;
  __shared__ int red[256];
  const DevParams<R>& p = *prm;
  const int tid = threadIdx.x;
  const int ntile = min(*count, cap);  // a list holds every tile at most once
  for (int it = blockIdx.x; it < ntile; it += gridDim.x) {
  const int tile = list[it];
  const int x0 = 3 + (tile / nty) * TX;  // first interior row of the tile (padded index)
  const int y0 = 3 + (tile % nty) * TY;
  int myflag = -2;

  // 1. stage phi (halo 2) and mu (halo 1); indices clamped into the padded array
  for (int i = tid; i < RX2 * RY2; i += 256) {
    int rx = i / RY2, ry = i % RY2;
    int gx = min(x0 - 2 + rx, p.rx - 1), gy = min(y0 - 2 + ry, p.ry - 1);
#pragma unroll
    for (int a = 0; a < P; a++) sm.phi[a][rx][ry] = phi[idx(p, a, gx, gy)];
  }
  for (int i = tid; i < RX1 * RY1; i += 256) {
    int rx = i / RY1, ry = i % RY1;
    int gx = min(x0 - 1 + rx, p.rx - 1), gy = min(y0 - 1 + ry, p.ry - 1);
#pragma unroll
    for (int k = 0; k < C; k++) sm.mu[k][rx][ry] = mu[idx(p, k, gx, gy)];
  }
  __syncthreads();

  // 2. delta-phi on the tile plus its 1-cell ring (region cell (rx,ry) is padded
  //    cell (x0-1+rx, y0-1+ry); its 3x3 phi block starts at phi region (rx, ry))
  for (int i = tid; i < RX1 * RY1; i += 256) {
    int rx = i / RY1, ry = i % RY1;
    R v[P][3][3];
#pragma unroll
    for (int a = 0; a < P; a++)
#pragma unroll
      for (int u = 0; u < 3; u++)
#pragma unroll
        for (int w = 0; w < 3; w++) v[a][u][w] = sm.phi[a][rx + u][ry + w];
    Nbhd<P, R> n;
    make_nbhd<P>(p, v, n);
    R m[C], dp[P];
#pragma unroll
    for (int k = 0; k < C; k++) m[k] = sm.mu[k][rx][ry];
    cell_dphi<P, C>(p, n, m, dp);
#pragma unroll
    for (int a = 0; a < P; a++) sm.dp[a][rx][ry] = dp[a];
  }
  __syncthreads();

  // 3. update of the tile cells
  for (int i = tid; i < TX * TY; i += 256) {
    int tx = i / TY, ty = i % TY;
    int x = x0 + tx, y = y0 + ty;
    if (x > p.mesh_x + 2 || y > p.mesh_y + 2) continue;
    const int ax = tx + 1, ay = ty + 1;  // position in the halo-1 regions
    R v[P][3][3];
#pragma unroll
    for (int a = 0; a < P; a++)
#pragma unroll
      for (int u = 0; u < 3; u++)
#pragma unroll
        for (int w = 0; w < 3; w++) v[a][u][w] = sm.phi[a][tx + 1 + u][ty + 1 + w];
    Nbhd<P, R> n;
    make_nbhd<P>(p, v, n);
    R phc[P], phf[P], phb[P], phr[P], phl[P], dc[P], df[P], db[P], dr[P], dl[P];
#pragma unroll
    for (int a = 0; a < P; a++) {
      phc[a] = v[a][1][1];
      phf[a] = v[a][2][1];
      phb[a] = v[a][0][1];
      phr[a] = v[a][1][2];
      phl[a] = v[a][1][0];
      dc[a] = sm.dp[a][ax][ay];
      df[a] = sm.dp[a][ax + 1][ay];
      db[a] = sm.dp[a][ax - 1][ay];
      dr[a] = sm.dp[a][ax][ay + 1];
      dl[a] = sm.dp[a][ax][ay - 1];
    }
    R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
    for (int k = 0; k < C; k++) {
      mc[k] = sm.mu[k][ax][ay];
      mf[k] = sm.mu[k][ax + 1][ay];
      mb[k] = sm.mu[k][ax - 1][ay];
      mr[k] = sm.mu[k][ax][ay + 1];
      ml[k] = sm.mu[k][ax][ay - 1];
    }
    R jf[C], jb[C], jr[C], jl[C];
    face_jat<P, C>(p, n.gXc, n.cYc, n.cYf, phc, phf, mc, mf, dc, df, true, jf);
    face_jat<P, C>(p, n.gXb, n.cYb, n.cYc, phb, phc, mb, mc, db, dc, true, jb);
    face_jat<P, C>(p, n.gYc, n.cXc, n.cXr, phc, phr, mc, mr, dc, dr, y != p.yskip, jr);
    face_jat<P, C>(p, n.gYl, n.cXl, n.cXc, phl, phc, ml, mc, dl, dc, (y - 1) != p.yskip, jl);
    R Dc[C][C], Df[C][C], Db[C][C], Dr[C][C], Dl[C][C];
    cell_D<P, C>(p, phc, Dc);
    cell_D<P, C>(p, phf, Df);
    cell_D<P, C>(p, phb, Db);
    cell_D<P, C>(p, phr, Dr);
    cell_D<P, C>(p, phl, Dl);
    R Dmf[C][C], Dmb[C][C], Dmr[C][C], Dml[C][C], gmf[C], gmb[C], gmr[C], gml[C];
#pragma unroll
    for (int k = 0; k < C; k++) {
#pragma unroll
      for (int l = 0; l < C; l++) {
        Dmf[k][l] = (Df[k][l] + Dc[k][l]) * R(0.5);
        Dmb[k][l] = (Dc[k][l] + Db[k][l]) * R(0.5);
        Dmr[k][l] = (Dr[k][l] + Dc[k][l]) * R(0.5);
        Dml[k][l] = (Dc[k][l] + Dl[k][l]) * R(0.5);
      }
      gmf[k] = div_dx(mf[k] - mc[k], p);
      gmb[k] = div_dx(mc[k] - mb[k], p);
      gmr[k] = div_dy(mr[k] - mc[k], p);
      gml[k] = div_dy(mc[k] - ml[k], p);
    }
    R pho[P], muo[C], dmu[C];
    cell_update<P, C>(p, phc, mc, dc, jf, jb, jr, jl, Dmf, Dmb, Dmr, Dml, gmf, gmb, gmr, gml, pho, muo, dmu);
    myflag = flag_combine(myflag, onehot_bits<P>(pho));
#pragma unroll
    for (int a = 0; a < P; a++) write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, pho[a]);
    if constexpr (Ops<R>::Exact) {
#pragma unroll
      for (int k = 0; k < C; k++) write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, muo[k]);
    } else {
      // compensated accumulation of the mu increment
#pragma unroll
      for (int k = 0; k < C; k++) {
        R lo = mulo[idx(p, k, x, y)];
        R yk = dmu[k] - lo;
        R t = mc[k] + yk;
        R lo_n = (t - mc[k]) - yk;
        write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, t);
        mulo_o[idx(p, k, x, y)] = lo_n;
      }
    }
  }
  int f = block_flag(myflag, red);
  if (tid == 0) flag_o[tile] = f == -2 ? -1 : f;
  }  // tile loop
}

// mu/phi update of a cell whose 3x3 block is one-hot in one phase and whose own
// and four neighbours' delta-phi are +0: the antitrapping fluxes and the dh/dt
// source are exact zeros and the five mobilities are equal, so the update is the
// bulk branch of cell_update with those zeros -- bit-identical to conc_cell.
// bulk_mu takes the cell's phase vector ph, writes mu (and the binary32 low
// parts) and returns the new phase vector in pho (ph + 0, the same bits).
// bulk_mu_v takes mu of the five-point stencil and the mobility Dm that the five
// cells share (they carry the same phi), and the phase tables from q (p, or a
// view of the cell's phase alone).
template <int P, int C, class R, bool NI = false, class Pm>
__device__ __forceinline__ void bulk_mu_v(const DevParams<R>& p, const Pm& q, const R* ph, const R (&Dm)[C][C],
                                          const R* mc, const R* mf, const R* mb, const R* mr, const R* ml,
                                          const R* __restrict__ mulo, R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                          int x, int y, R T, R* pho, const R* lo_pre = nullptr) {
  R zp[P], z[C];
#pragma unroll
  for (int a = 0; a < P; a++) zp[a] = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) z[k] = R(0);
  R gmf[C], gmb[C], gmr[C], gml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    gmf[k] = div_dx(mf[k] - mc[k], p);
    gmb[k] = div_dx(mc[k] - mb[k], p);
    gmr[k] = div_dy(mr[k] - mc[k], p);
    gml[k] = div_dy(mc[k] - ml[k], p);
  }
  R muo[C], dmu[C];
  cell_update<P, C, R, NI>(q, ph, mc, zp, z, z, z, z, Dm, Dm, Dm, Dm, gmf, gmb, gmr, gml, pho, muo, dmu, T);
  if constexpr (Ops<R>::Exact) {
#pragma unroll
    for (int k = 0; k < C; k++) write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, muo[k]);
  } else {
#pragma unroll
    for (int k = 0; k < C; k++) {
      R lo = lo_pre ? lo_pre[k] : mulo[idx(p, k, x, y)];
      R yk = dmu[k] - lo;
      R t = mc[k] + yk;
      R lo_n = (t - mc[k]) - yk;
      write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, t);
      mulo_o[idx(p, k, x, y)] = lo_n;
    }
  }
}

template <int P, int C, class R, bool NI = false>
__device__ __forceinline__ void bulk_mu(const DevParams<R>& p, const R* ph, const R* __restrict__ mu,
                                        const R* __restrict__ mulo, R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                        int x, int y, R T, R* pho) {
  R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    mc[k] = mu[idx(p, k, x, y)];
    mf[k] = mu[idx(p, k, x + 1, y)];
    mb[k] = mu[idx(p, k, x - 1, y)];
    mr[k] = mu[idx(p, k, x, y + 1)];
    ml[k] = mu[idx(p, k, x, y - 1)];
  }
  R D[C][C], Dm[C][C];
  cell_D<P, C>(p, ph, D);
#pragma unroll
  for (int k = 0; k < C; k++)
#pragma unroll
    for (int l = 0; l < C; l++) Dm[k][l] = (D[k][l] + D[k][l]) * R(0.5);
  bulk_mu_v<P, C, R, NI>(p, p, ph, Dm, mc, mf, mb, mr, ml, mulo, mu_o, mulo_o, x, y, T, pho);
}

// bulk_mu_v of a cell at the exact one-hot vector of phase a: that phase's tables
// alone, and its mobility from the table formed on the host (Dm_bulk, the same
// values).
template <int C, class R, bool NI = false>
__device__ __forceinline__ void bulk_mu_onehot(const DevParams<R>& p, int a, const R* mc, const R* mf, const R* mb,
                                               const R* mr, const R* ml, const R* __restrict__ mulo,
                                               R* __restrict__ mu_o, R* __restrict__ mulo_o, int x, int y, R T,
                                               const R* lo_pre = nullptr) {
  const PhaseParams<R> q(p, a);
  const R one[1] = {R(1.0)};
  R Dm[C][C], pho[1];
#pragma unroll
  for (int k = 0; k < C; k++)
#pragma unroll
    for (int l = 0; l < C; l++) Dm[k][l] = p.Dm_bulk[a][k][l];
  bulk_mu_v<1, C, R, NI>(p, q, one, Dm, mc, mf, mb, mr, ml, mulo, mu_o, mulo_o, x, y, T, pho, lo_pre);
}

template <int P, int C, class R, bool NI = false>
__device__ __forceinline__ void bulk_cell(const DevParams<R>& p, const R* __restrict__ phi, const R* __restrict__ mu,
                                          const R* __restrict__ mulo, R* __restrict__ phi_o, R* __restrict__ mu_o,
                                          R* __restrict__ mulo_o, int x, int y, R T = R(0)) {
  R ph[P], pho[P];
#pragma unroll
  for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, x, y)];
  bulk_mu<P, C, R, NI>(p, ph, mu, mulo, mu_o, mulo_o, x, y, T, pho);
#pragma unroll
  for (int a = 0; a < P; a++) write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, pho[a]);
}

// Bulk tiles: the tile and its 2-cell halo hold the exact one-hot vector of
// phase flag_i (onehot_bits), so every cell satisfies the bulk_cell conditions.
// The phase vector is known from the flag: phi is not read, and its planes are
// written only where the output buffer does not hold the same vector already, at
// the cells and at their ghost images (flag_o describes the state of two steps
// back until it is overwritten here; the sweeps that set it write both, k_flags
// looks at both).
// The sweep moves the mu planes alone: on 64 grids of 64^2 to 512^2 (two phases,
// binary64) 143 -> 58 us a step.  That is 100 MB at 1.7 TB/s, below half of a
// large copy's rate; what bounds it is not known (reading the next tile's list
// entry, grid and flags ahead of the current tile's update changed nothing).
template <int P, int C, class R, int TX, int TY>
__global__ void __launch_bounds__(256) k_bulk(const Inst<R>* __restrict__ inst, const int* __restrict__ tinst, int par,
                                              const int* __restrict__ list, const int* __restrict__ count,
                                              const int* __restrict__ flag_i, int* __restrict__ flag_o, int cap) {
  const int ntile = min(*count, cap);  // a list holds every tile at most once
  for (int it = blockIdx.x; it < ntile; it += gridDim.x) {
    const int tile = list[it];
    const Inst<R>& g = inst_of(inst, tinst, tile);
    const DevParams<R>& p = *g.prm;
    const int lt = tile - g.tile0;
    const int x0 = 3 + (lt / g.nty) * TX;
    const int y0 = 3 + (lt % g.nty) * TY;
    const R *phi = g.phi[par], *mu = g.mu[par], *mulo = g.mulo[par];
    R *phi_o = g.phi[par ^ 1], *mu_o = g.mu[par ^ 1], *mulo_o = g.mulo[par ^ 1];
    const int f = flag_i[tile];
    const bool held = flag_o[tile] == f;
    for (int i = threadIdx.x; i < TX * TY; i += 256) {
      const int x = x0 + i / TY, y = y0 + i % TY;
      if (x > p.mesh_x + 2 || y > p.mesh_y + 2) continue;
      R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
      for (int k = 0; k < C; k++) {
        mc[k] = mu[idx(p, k, x, y)];
        mf[k] = mu[idx(p, k, x + 1, y)];
        mb[k] = mu[idx(p, k, x - 1, y)];
        mr[k] = mu[idx(p, k, x, y + 1)];
        ml[k] = mu[idx(p, k, x, y - 1)];
      }
      bulk_mu_onehot<C, R>(p, f, mc, mf, mb, mr, ml, mulo, mu_o, mulo_o, x, y, R(0));
      if (!held) {  // the same bits as ph + 0
#pragma unroll
        for (int a = 0; a < P; a++)
          write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, a == f ? R(1.0) : R(0));
      }
    }
    __syncthreads();  // flag_o[tile] has been read
    if (threadIdx.x == 0) flag_o[tile] = f;
  }
}

// Interface-cell test of the phase sweep: some phase has a non-zero divergence
// (the activity test of cell_dphi, same expressions).  Cells that fail it get
// delta-phi from the projection alone.
template <int P, class R>
__device__ __forceinline__ bool phase_active(const DevParams<R>& p, const R* __restrict__ phi, int x, int y, R* ph) {
  bool any = false;
#pragma unroll
  for (int a = 0; a < P; a++) {
    const R c = phi[idx(p, a, x, y)];
    const R gxc = div_dx(phi[idx(p, a, x + 1, y)] - c, p), gxb = div_dx(c - phi[idx(p, a, x - 1, y)], p);
    const R gyc = div_dy(phi[idx(p, a, x, y + 1)] - c, p), gyl = div_dy(c - phi[idx(p, a, x, y - 1)], p);
    R d = div_dx(gxc - gxb, p);
    d += div_dy(gyc - gyl, p);
    any = any || fabs(d) > R(0);
    ph[a] = c;
  }
  return any;
}

// Uniform 5-point neighbourhood in every phase: then every gradient of the
// phase sweep is an exact zero, so no phase is active.  A conservative form of
// phase_active without arithmetic (all loads first, then comparisons): a cell
// that fails it goes to the dense kernel, which decides activity exactly.
template <int P, class R>
__device__ __forceinline__ bool phase_uniform(const DevParams<R>& p, const R* __restrict__ phi, int x, int y, R* ph) {
  R c[P], f[P], b[P], r[P], l[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    c[a] = phi[idx(p, a, x, y)];
    f[a] = phi[idx(p, a, x + 1, y)];
    b[a] = phi[idx(p, a, x - 1, y)];
    r[a] = phi[idx(p, a, x, y + 1)];
    l[a] = phi[idx(p, a, x, y - 1)];
  }
  bool u = true;
#pragma unroll
  for (int a = 0; a < P; a++) {
    u = u && f[a] == c[a] && b[a] == c[a] && r[a] == c[a] && l[a] == c[a];
    ph[a] = c[a];
  }
  return u;
}

// Split two-pass step (path 4).  The dense two-pass kernels need about 240
// registers per lane for interface cells, which leaves two waves per SIMD also
// for bulk cells, whose few loads then go unhidden.  Each sweep of a split step
// is a light kernel over the full grid, with the block shape of the dense
// kernel, that finishes every cell with an exact shortcut -- phase sweep: no
// active phase, delta-phi from the projection alone; mu sweep: bulk_cell,
// decided on the codes of the 3x3 block -- and appends each block holding any
// other cell to a list; the dense kernel then runs over the listed blocks only
// and recomputes all their cells (the shortcuts are bit-identical to the full
// arithmetic).  Counters: cnt[0] (phase list) is cleared by the mu-sweep light
// kernel, cnt[1] (mu list) by the next phase-sweep light kernel, each after
// the kernel that read it has finished.
template <int P, class R>
__global__ void __launch_bounds__(BX * BY) k_phase_split(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                         R* __restrict__ dphi, signed char* __restrict__ code,
                                                         int* __restrict__ list, int* __restrict__ cnt) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 2 + bx * BX + threadIdx.x;
  const int x = 2 + by * BY + threadIdx.y;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && threadIdx.y == 0) cnt[1] = 0;
  int heavy = 0;
  if (x <= p.rx - 3 && y <= p.ry - 3) {
    R ph[P];
    if (!phase_uniform<P>(p, phi, x, y, ph)) {  // possibly active: the dense kernel decides
      heavy = 1;
      code[(size_t)x * p.pitch + y] = -1;
    } else {
      R dp[P];
      bool act[P];
#pragma unroll
      for (int a = 0; a < P; a++) {
        dp[a] = R(0);
        act[a] = false;
      }
      project_simplex<P>(ph, act, dp);
      bool zero = true;
#pragma unroll
      for (int a = 0; a < P; a++) zero = zero && dp[a] == R(0) && !signbit(dp[a]);
      const int cd = zero ? onehot_phase<P>(ph) : -1;
      code[(size_t)x * p.pitch + y] = (signed char)cd;
      if (cd < 0) {  // a code >= 0 stands for delta-phi +0 (load_dphi); the planes are left as they are
#pragma unroll
        for (int a = 0; a < P; a++) dphi[idx(p, a, x, y)] = dp[a];
      }
    }
  }
  if (__syncthreads_or(heavy) && threadIdx.x == 0 && threadIdx.y == 0) {
    const int slot = atomicAdd(&cnt[0], 1);
    if (slot < (int)(gridDim.x * gridDim.y)) list[slot] = by * gridDim.x + bx;  // a list holds every block at most
  }
}

// mu sweep of a split step: the cells (block shape of k_conc_lds / k_conc_march
// with one row per wave) whose 3x3 block carries one code a >= 0 take bulk_cell.
// With NI, at the row temperature the dense kernel uses (tb, tsh as there).
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) k_conc_split(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                        const R* __restrict__ mu, const R* __restrict__ mulo,
                                                        const signed char* __restrict__ code, R* __restrict__ phi_o,
                                                        R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                                        int* __restrict__ list, int* __restrict__ cnt, R tb = R(0),
                                                        int tsh = 0) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int lane = threadIdx.x;
  const int y = 2 + bx * MW + lane;  // lane 0 sits one column before the block's cells, as in k_conc_lds
  const int x = 3 + by * BY + threadIdx.y;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && threadIdx.y == 0) cnt[0] = 0;
  int heavy = 0;
  if (lane > 0 && x <= p.mesh_x + 2 && y <= p.mesh_y + 2) {
    int cc = code[(size_t)x * p.pitch + y];
#pragma unroll
    for (int u = -1; u <= 1; u++)
#pragma unroll
      for (int w = -1; w <= 1; w++) cc = code[(size_t)(x + u) * p.pitch + y + w] == cc ? cc : -1;
    if (cc >= 0) bulk_cell<P, C, R, NI>(p, phi, mu, mulo, phi_o, mu_o, mulo_o, x, y, NI ? temp_row(p, tb, y, true, tsh) : R(0));
    else heavy = 1;
  }
  if (__syncthreads_or(heavy) && threadIdx.x == 0 && threadIdx.y == 0) {
    const int slot = atomicAdd(&cnt[1], 1);
    if (slot < (int)(gridDim.x * gridDim.y)) list[slot] = by * gridDim.x + bx;
  }
}

// Compact split step (path 5).  The light kernels of the split step decide
// per cell, as there, which cells an exact shortcut finishes; every other cell
// is appended to a grid-wide cell list, and the dense kernels then run one
// listed cell per lane.  The block lists of path 4 make the dense kernels
// recompute every cell of a block that holds one interface cell, and a wave of
// 64 columns of one row then carries few interface lanes: on the 4-phase
// 1024^2 seeded grid, 2% of the cells need the dense arithmetic, the listed
// blocks hold 4.5 times as many cells, and a wave that computes any of them
// has a quarter of its lanes busy.  Listed cells keep the row order of the
// light blocks that appended them (one atomic per block, consecutive slots for
// its waves and lanes), so the dense kernels' stencil loads stay mostly
// coalesced.  One atomic per wave instead serialises some two thousand
// device-scope atomics on one counter per launch on that grid, which doubled
// the light kernels' time.
//
// A list entry is (x << 16) | y (padded indices below 65536).  Every thread
// of the block (BX x BY, one wave per threadIdx.y) calls it.
static_assert(BX == 64, "cell_append takes threadIdx.x for the lane and threadIdx.y for the wave");
__device__ __forceinline__ void cell_append(bool want, int x, int y, int* __restrict__ list, int* __restrict__ cnt,
                                            int cap) {
  __shared__ int wn[BY + 1];
  const unsigned long long m = __ballot(want);
  const int lane = threadIdx.x, w = threadIdx.y;
  if (lane == 0) wn[w] = __popcll(m);
  __syncthreads();
  if (lane == 0 && w == 0) {
    int t = 0;
#pragma unroll
    for (int i = 0; i < BY; i++) {
      const int v = wn[i];
      wn[i] = t;
      t += v;
    }
    wn[BY] = t ? atomicAdd(cnt, t) : 0;
  }
  __syncthreads();
  if (want) {
    const int s = wn[BY] + wn[w] + __popcll(m & ((1ull << lane) - 1ull));
    if (s < cap) list[s] = (x << 16) | y;  // a list holds every cell at most once
  }
}

// Light phase sweep of path 5 over [2, rows-3]^2 (k_phase_split with a cell
// list).  Clears the mu-sweep counter cnt[1], which the previous step's dense
// kernel has finished reading.
template <int P, class R>
__global__ void __launch_bounds__(BX * BY) k_phase_light(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                         R* __restrict__ dphi, signed char* __restrict__ code,
                                                         int* __restrict__ list, int* __restrict__ cnt, int cap) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 2 + bx * BX + threadIdx.x;
  const int x = 2 + by * BY + threadIdx.y;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && threadIdx.y == 0) cnt[1] = 0;
  bool heavy = false;
  if (x <= p.rx - 3 && y <= p.ry - 3) {
    R ph[P];
    if (!phase_uniform<P>(p, phi, x, y, ph)) {  // possibly active: the dense kernel decides
      heavy = true;
      code[(size_t)x * p.pitch + y] = -1;
    } else {
      R dp[P];
      bool act[P];
#pragma unroll
      for (int a = 0; a < P; a++) {
        dp[a] = R(0);
        act[a] = false;
      }
      project_simplex<P>(ph, act, dp);
      bool zero = true;
#pragma unroll
      for (int a = 0; a < P; a++) zero = zero && dp[a] == R(0) && !signbit(dp[a]);
      const int cd = zero ? onehot_phase<P>(ph) : -1;
      code[(size_t)x * p.pitch + y] = (signed char)cd;
      if (cd < 0) {  // a code >= 0 stands for delta-phi +0 (load_dphi); the planes are left as they are
#pragma unroll
        for (int a = 0; a < P; a++) dphi[idx(p, a, x, y)] = dp[a];
      }
    }
  }
  cell_append(heavy, x, y, list, cnt, cap);
}

// Dense phase sweep of path 5: delta-phi of listed cell i = blockIdx.x * 256 +
// threadIdx.x, in a grid-stride loop over the list.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(256) GP_HEAVY k_phase_cells(const DevParams<R>* __restrict__ prm,
                                                              const R* __restrict__ phi, const R* __restrict__ mu,
                                                              R* __restrict__ dphi, R tb, int tmode,
                                                              const int* __restrict__ list,
                                                              const int* __restrict__ cnt, int cap,
                                                              NoiseRef nz) {
  const DevParams<R>& p = *prm;
  const int n = min(*cnt, cap);
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int e = list[i], x = e >> 16, y = e & 0xffff;
    if (x < 2 || x > p.rx - 3 || y < 2 || y > p.ry - 3) continue;  // entries are cells of the phase sweep
    phase_cell<P, C, R, NI>(p, phi, mu, dphi, x, y, NI ? temp_row(p, tb, y, (tmode & 1) != 0, tmode >> 1) : R(0),
                            nz);
  }
}

// Light mu sweep of path 5 over the interior, 64 columns per wave: a cell
// whose 3x3 block carries one code a >= 0 takes bulk_cell, any other is
// listed.  The phase-sweep counter cnt[0] is cleared by k_conc_cells.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) k_conc_light(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                        const R* __restrict__ mu, const R* __restrict__ mulo,
                                                        const signed char* __restrict__ code, R* __restrict__ phi_o,
                                                        R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                                        int* __restrict__ list, int* __restrict__ cnt, int cap, R tb,
                                                        int tsh) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 3 + bx * BX + threadIdx.x;
  const int x = 3 + by * BY + threadIdx.y;
  bool heavy = false;
  if (x <= p.mesh_x + 2 && y <= p.mesh_y + 2) {
    int cc = code[(size_t)x * p.pitch + y];
#pragma unroll
    for (int u = -1; u <= 1; u++)
#pragma unroll
      for (int w = -1; w <= 1; w++) cc = code[(size_t)(x + u) * p.pitch + y + w] == cc ? cc : -1;
    if (cc >= 0) bulk_cell<P, C, R, NI>(p, phi, mu, mulo, phi_o, mu_o, mulo_o, x, y, NI ? temp_row(p, tb, y, true, tsh) : R(0));
    else heavy = true;
  }
  cell_append(heavy, x, y, list, cnt + 1, cap);
}

// Dense mu update of interior cell (x, y) for the compact split and one-hot
// paths, with all four antitrapping faces evaluated by its own lane (face_jat
// is the same function of the same operands whichever cell of a face
// evaluates it, so the result is the shared-face kernels' bit for bit);
// delta-phi is read through the codes.  With oh_o (path 6) it also writes the
// exact one-hot code of the cell's new phi there.
template <int P, int C, class R, bool NI = false>
__device__ __forceinline__ void conc_cell_dense(const DevParams<R>& p, const R* __restrict__ phi,
                                                const R* __restrict__ mu, const R* __restrict__ dphi,
                                                const R* __restrict__ mulo, R* __restrict__ phi_o,
                                                R* __restrict__ mu_o, R* __restrict__ mulo_o, R tb, int tsh,
                                                const signed char* __restrict__ code, signed char* __restrict__ oh_o,
                                                int x, int y) {
  const R Tc = NI ? temp_row(p, tb, y, true, tsh) : R(0);
  const R Tr = NI ? temp_row(p, tb, y + 1, true, tsh) : R(0);
  const R Tl = NI ? temp_row(p, tb, y - 1, true, tsh) : R(0);
  R v[P][3][3];
  load3x3<P>(p, phi, x, y, v);
  Nbhd<P, R> nb;
  make_nbhd<P>(p, v, nb);
  R phc[P], phf[P], phb[P], phr[P], phl[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    phc[a] = v[a][1][1];
    phf[a] = v[a][2][1];
    phb[a] = v[a][0][1];
    phr[a] = v[a][1][2];
    phl[a] = v[a][1][0];
  }
  R dc[P], df[P], db[P], dr[P], dl[P];
  load_dphi<P>(p, dphi, code, x, y, dc);
  load_dphi<P>(p, dphi, code, x + 1, y, df);
  load_dphi<P>(p, dphi, code, x - 1, y, db);
  load_dphi<P>(p, dphi, code, x, y + 1, dr);
  load_dphi<P>(p, dphi, code, x, y - 1, dl);
  R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    mc[k] = mu[idx(p, k, x, y)];
    mf[k] = mu[idx(p, k, x + 1, y)];
    mb[k] = mu[idx(p, k, x - 1, y)];
    mr[k] = mu[idx(p, k, x, y + 1)];
    ml[k] = mu[idx(p, k, x, y - 1)];
  }
  R jf[C], jb[C], jr[C], jl[C];
  face_jat<P, C, R, NI>(p, nb.gXc, nb.cYc, nb.cYf, phc, phf, mc, mf, dc, df, true, jf, Tc, Tc);
  face_jat<P, C, R, NI>(p, nb.gXb, nb.cYb, nb.cYc, phb, phc, mb, mc, db, dc, true, jb, Tc, Tc);
  face_jat<P, C, R, NI>(p, nb.gYc, nb.cXc, nb.cXr, phc, phr, mc, mr, dc, dr, y != p.yskip, jr, Tc, Tr);
  face_jat<P, C, R, NI>(p, nb.gYl, nb.cXl, nb.cXc, phl, phc, ml, mc, dl, dc, (y - 1) != p.yskip, jl, Tl, Tc);
  conc_apply<P, C, R, !Ops<R>::Exact, NI>(p, v, mc, mf, mb, mr, ml, dc, jf, jb, jr, jl, mulo, phi_o, mu_o, mulo_o, x,
                                         y, Tc);
  if (oh_o) {  // the exact one-hot code of the new phi (phc + dc, the value written)
    R pn[P];
#pragma unroll
    for (int a = 0; a < P; a++) pn[a] = phc[a] + dc[a];
    oh_o[(size_t)x * p.pitch + y] = (signed char)onehot_bits<P>(pn);
  }
}

// Dense mu sweep of path 5: conc_cell_dense on listed cell i = blockIdx.x *
// 256 + threadIdx.x, in a grid-stride loop over the list.  Reads the mu-sweep
// counter cnt[1] and clears the phase-sweep counter cnt[0], whose readers
// (k_phase_cells) have finished.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(256) GP_HEAVY k_conc_cells(const DevParams<R>* __restrict__ prm,
                                                             const R* __restrict__ phi, const R* __restrict__ mu,
                                                             const R* __restrict__ dphi, const R* __restrict__ mulo,
                                                             R* __restrict__ phi_o, R* __restrict__ mu_o,
                                                             R* __restrict__ mulo_o, R tb, int tsh,
                                                             const int* __restrict__ list, int* __restrict__ cnt,
                                                             int cap, const signed char* __restrict__ code) {
  const DevParams<R>& p = *prm;
  const int n = min(cnt[1], cap);
  if (blockIdx.x == 0 && threadIdx.x == 0) cnt[0] = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int e = list[i], x = e >> 16, y = e & 0xffff;
    if (x < 3 || x > p.mesh_x + 2 || y < 3 || y > p.mesh_y + 2) continue;  // entries are interior cells
    conc_cell_dense<P, C, R, NI>(p, phi, mu, dphi, mulo, phi_o, mu_o, mulo_o, tb, tsh, code,
                                 (signed char*)nullptr, x, y);
  }
}

// One-hot path (path 6): path 5's sweeps with one byte plane per state
// buffer, oh[b], where oh[b][c] = a >= 0 says that buffer b holds the exact
// one-hot vector of phase a at cell c (and at its ghost images).  With them
// the light phase sweep gives a cell whose five-point cross carries one such a
// the code a without loading phi (phase_uniform holds there and the projection
// of a one-hot vector is +0), and the light mu sweep takes a bulk cell's phase
// vector from its code instead of loading it and leaves its phi planes
// unwritten when the output buffer already holds that one-hot vector (the
// state two steps back, unchanged since).  Path 6's codes stand for the exact
// one-hot bits (onehot_bits), so that a code gives the phase vector itself.
// The dense phase sweep and the light mu sweep run as one launch: neither
// reads what the other writes, and the dense waves, bound by the latency of
// one cell's arithmetic, then overlap the light ones.
//
// Its cell lists are segmented: a light block with hardware linear index L
// appends to segment L mod kSegs through that segment's counter, so the
// appending blocks of a launch spread their device-scope atomics over kSegs
// addresses instead of queueing on one (such atomics serialise at about 12 ns
// each per address on MI355X: one per block of a 1024^2 sweep on 8 addresses
// cost 8 us).  Segment k holds every cell of the blocks of its class (those of
// a launch with index = k mod kSegs), so it cannot overflow; the counters sit
// kSegStride ints apart, and a dense lane finds listed cell i by walking the
// kSegs counts.  kSegs is a multiple of 8, so a segment's blocks share an XCD;
// 32 segments made the dense kernels, which walk the counts, 5-10% slower and
// the light kernels no faster.
constexpr int kSegs = 8;
constexpr int kSegStride = 32;
constexpr int kSegInts = 2 * kSegs * kSegStride;  // phase-sweep counters, then mu-sweep counters

// Cells per block of the light mu sweep and of the light phase sweep (kPhaseCols
// columns per lane).
constexpr int kMuCells = BX * BY;
constexpr int kPhaseCols = 4;
constexpr int kPhaseCells = BX * BY * kPhaseCols;

// First slot of segment k of a list written by a launch of nblk blocks of
// `cells` cells.
template <int cells>
__host__ __device__ __forceinline__ int seg_base(int k, int nblk) {
  const int q = nblk / kSegs, r = nblk % kSegs;
  return (k * q + (k < r ? k : r)) * cells;
}

// Grid of the light phase sweep over [2, rows-3]^2: groups of kPhaseCols
// columns from column 0 on (a group is one aligned word of the byte planes).
__host__ __device__ inline dim3 phase_light_grid(int rx, int ry) {
  return dim3(((ry - 2 + kPhaseCols - 1) / kPhaseCols + BX - 1) / BX, (rx - 4 + BY - 1) / BY);
}

// cell_append into segment L mod kSegs (cnt: the list's kSegs counters) of a
// list whose blocks hold `cells` cells each.
template <int cells>
__device__ __forceinline__ void cell_append_seg(bool want, int x, int y, int L, int nblk, int* __restrict__ list,
                                                int* __restrict__ cnt) {
  __shared__ int wn[BY + 1];
  const unsigned long long m = __ballot(want);
  const int lane = threadIdx.x, w = threadIdx.y;
  if (lane == 0) wn[w] = __popcll(m);
  __syncthreads();
  if (lane == 0 && w == 0) {
    int t = 0;
#pragma unroll
    for (int i = 0; i < BY; i++) {
      const int v = wn[i];
      wn[i] = t;
      t += v;
    }
    wn[BY] = t ? atomicAdd(cnt + kSegStride * (L % kSegs), t) : 0;
  }
  __syncthreads();
  if (want)
    list[seg_base<cells>(L % kSegs, nblk) + wn[BY] + wn[w] + __popcll(m & ((1ull << lane) - 1ull))] = (x << 16) | y;
}

// Listed cells of a segmented list: n = their number; cell i (< n) is entry
// seg_at(i) of the list.
template <int cells>
struct SegList {
  int c[kSegs], n, nblk;
  __device__ __forceinline__ SegList(const int* __restrict__ cnt, int nblk_) : n(0), nblk(nblk_) {
#pragma unroll
    for (int k = 0; k < kSegs; k++) {
      const int q = nblk / kSegs, r = nblk % kSegs;
      c[k] = min(cnt[kSegStride * k], (q + (k < r ? 1 : 0)) * cells);  // a segment holds at most its capacity
      n += c[k];
    }
  }
  __device__ __forceinline__ int seg_at(int i) const {
    int k = 0;
#pragma unroll
    for (int j = 0; j < kSegs - 1; j++)
      if (k == j && i >= c[j]) {
        i -= c[j];
        k = j + 1;
      }
    return seg_base<cells>(k, nblk) + i;
  }
};

// oh of the current buffer from its interior cells, oh of the other buffer
// unknown (-1): the set-up after a step of another path or a new state.  A
// cell that may have ghost images (outside the band that is the source of none:
// the copies of Neumann and periodic faces reach the fourth row from the face)
// is left unknown, so that only a write of the cell and its images by this
// path's own sweeps vouches for them.
template <int P, class R>
__global__ void __launch_bounds__(BX * BY) k_oh_prime(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                      signed char* __restrict__ oh, signed char* __restrict__ oh_x) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 3 + bx * BX + threadIdx.x;
  const int x = 3 + by * BY + threadIdx.y;
  if (x > p.mesh_x + 2 || y > p.mesh_y + 2) return;
  R ph[P];
#pragma unroll
  for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, x, y)];
  const size_t i = (size_t)x * p.pitch + y;
  const bool edge = x < p.gfree[0][0][0] || x > p.gfree[0][0][1] || y < p.gfree[0][1][0] || y > p.gfree[0][1][1];
  oh[i] = (signed char)(edge ? -1 : onehot_bits<P>(ph));
  oh_x[i] = -1;
}

// Counters of a segmented list pair, cleared (the set-up of a new buffer).
template <int Unused = 0>
__global__ void k_clear_seg(int* __restrict__ cnt) {
  for (int i = threadIdx.x; i < kSegInts; i += blockDim.x) cnt[i] = 0;
}

// phase_uniform, four phases at a time (with the loads of all nine in flight
// the light phase sweep took 240 registers), a wave leaving when none of its
// cells can still be uniform; ph is set where the result is true.
template <int P, class R>
__device__ __forceinline__ bool phase_uniform_by4(const DevParams<R>& p, const R* __restrict__ phi, int x, int y,
                                                  R* ph) {
  bool u = true;
#pragma unroll 1
  for (int a0 = 0; a0 < P && u; a0 += 4) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int a = a0 + j;
      if (P % 4 != 0 && a >= P) break;
      const R c = phi[idx(p, a, x, y)];
      const R f = phi[idx(p, a, x + 1, y)], b = phi[idx(p, a, x - 1, y)];
      const R r = phi[idx(p, a, x, y + 1)], l = phi[idx(p, a, x, y - 1)];
      u &= (f == c) & (b == c) & (r == c) & (l == c);
    }
  }
  if (u) {
#pragma unroll
    for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, x, y)];
  }
  return u;
}

// Light phase sweep of path 6 over [2, rows-3]^2: k_phase_light with the
// one-hot shortcut of the current buffer's plane oh, appending to the
// segmented phase-sweep list (lists + kSegInts, counters lists[0..]).  Clears
// the mu-sweep counters, which the previous step's dense kernel has finished
// reading.
//
// Almost every cell takes the shortcut, so the sweep is bound by the number of
// waves and of appends, not by its two bytes per cell: a lane first takes the
// kPhaseCols columns of one aligned word of the byte planes, and compares the
// words of the row, of the rows beside it and of the columns beside it.  The
// block's cells that fail (and those outside [4, mesh + 1]^2, whose cross
// leaves the interior) are gathered in LDS and looked at one per lane: left to
// the lane that found them, they ran one after another, and the sweep took 3-4
// times as long on states with wide interfaces.  One column per lane against
// this: 8.8 -> 6.3 us at 1024^2 and four phases, 17.6 -> 11.4 us at 1531 x 1021
// and six, 117 -> 70 us (binary32: 116 -> 63 us) at 4096^2 and nine.
template <int P, class R>
__global__ void __launch_bounds__(BX * BY) k_phase_light_oh(const DevParams<R>* __restrict__ prm,
                                                            const R* __restrict__ phi,
                                                            const signed char* __restrict__ oh, R* __restrict__ dphi,
                                                            signed char* __restrict__ code, int* __restrict__ lists) {
  static_assert(kPhaseCols == 4, "a group is one 32-bit word");
  __shared__ short todo[kPhaseCells];  // row of the block << 8 | column of the block
  __shared__ int tn[BY];
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int yb = bx * BX * kPhaseCols, xb = 2 + by * BY;
  const int y0 = yb + threadIdx.x * kPhaseCols, x = xb + threadIdx.y;
  const int L = blockIdx.y * gridDim.x + blockIdx.x, nblk = gridDim.x * gridDim.y;
  if (L == 0 && threadIdx.y == 0 && threadIdx.x < kSegs) lists[kSegs * kSegStride + kSegStride * threadIdx.x] = 0;
  unsigned left = 0;  // bit j: cell j is looked at
  if (x <= p.rx - 3 && y0 <= p.ry - 3) {
    const size_t i = (size_t)x * p.pitch + y0;  // pitch and y0 are multiples of 4
    unsigned sure = 0, w = 0;                   // bit 8 j + 7: cell j takes the shortcut; the codes
    if (x >= 4 && x <= p.mesh_x + 1) {
      w = *(const unsigned*)(oh + i);
      const unsigned u = *(const unsigned*)(oh + i + p.pitch), d = *(const unsigned*)(oh + i - p.pitch);
      const unsigned l = y0 ? (unsigned char)oh[i - 1] : 0, r = y0 + 4 < p.pitch ? (unsigned char)oh[i + 4] : 0;
      const unsigned t = (w ^ u) | (w ^ d) | (w ^ (w << 8 | l)) | (w ^ (w >> 8 | r << 24)) | (w & 0x80808080u);
      sure = ~(((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t) & 0x80808080u;  // bytes of t that are zero
#pragma unroll
      for (int j = 0; j < kPhaseCols; j++)
        if (y0 + j < 4 || y0 + j > p.mesh_y + 1) sure &= ~(0x80u << (8 * j));
    }
    if (sure == 0x80808080u) {
      *(unsigned*)(code + i) = w;
    } else {
#pragma unroll
      for (int j = 0; j < kPhaseCols; j++) {
        if (y0 + j < 2 || y0 + j > p.ry - 3) continue;
        if ((sure >> (8 * j + 7)) & 1) code[i + j] = (signed char)(w >> (8 * j));
        else left |= 1u << j;
      }
    }
  }
  // the cells left, in the order of the rows and columns
  int below = 0, all = 0;
#pragma unroll
  for (int j = 0; j < kPhaseCols; j++) {
    const unsigned long long m = __ballot((left >> j) & 1);
    below += __popcll(m & ((1ull << threadIdx.x) - 1ull));
    all += __popcll(m);
  }
  if (threadIdx.x == 0) tn[threadIdx.y] = all;
  __syncthreads();
  int n = 0;
#pragma unroll
  for (int i = 0; i < BY; i++) {
    if (i < (int)threadIdx.y) below += tn[i];
    n += tn[i];
  }
#pragma unroll
  for (int j = 0; j < kPhaseCols; j++)
    if ((left >> j) & 1) todo[below++] = (short)(threadIdx.y << 8 | (threadIdx.x * kPhaseCols + j));
  __syncthreads();
  for (int base = 0; base < n; base += BX * BY) {  // the same passes for every lane of the block
    const int k = base + (int)threadIdx.y * BX + (int)threadIdx.x;
    bool heavy = false;
    int cx = 0, cy = 0;
    if (k < n) {
      cx = xb + (todo[k] >> 8);
      cy = yb + (todo[k] & 0xff);
      signed char* cd_o = code + (size_t)cx * p.pitch + cy;
      R ph[P];
      if (!phase_uniform_by4<P>(p, phi, cx, cy, ph)) {  // possibly active: the dense kernel decides
        heavy = true;
        *cd_o = -1;
      } else {
        R dp[P];
        bool act[P];
#pragma unroll
        for (int a = 0; a < P; a++) {
          dp[a] = R(0);
          act[a] = false;
        }
        project_simplex<P>(ph, act, dp);
        bool zero = true;
#pragma unroll
        for (int a = 0; a < P; a++) zero = zero && dp[a] == R(0) && !signbit(dp[a]);
        const int cd = zero ? onehot_bits<P>(ph) : -1;
        *cd_o = (signed char)cd;
        if (cd < 0) {
#pragma unroll
          for (int a = 0; a < P; a++) dphi[idx(p, a, cx, cy)] = dp[a];
        }
      }
    }
    cell_append_seg<kPhaseCells>(heavy, cx, cy, L, nblk, lists + kSegInts, lists);
  }
}

// Light mu update of path 6 for one interior cell, in two halves: load()
// issues every load of the cell (codes, oh_o, mu, the binary32 low parts) and
// returns whether the dense sweep must take the cell (its 3x3 codes do not
// carry one a >= 0); finish() then applies bulk_mu_v with the phase vector
// from the code, writing the phi planes only where oh_o differs.
template <int P, int C, class R, bool NI>
struct LightMu {
  R mc[C], mf[C], mb[C], mr[C], ml[C], lo[C];
  int cc, oo;
  __device__ __forceinline__ bool load(const DevParams<R>& p, int x, int y, const R* __restrict__ mu,
                                       const R* __restrict__ mulo, const signed char* __restrict__ code,
                                       const signed char* __restrict__ oh_o) {
    const size_t i = (size_t)x * p.pitch + y;
    signed char cd[3][3];
#pragma unroll
    for (int u = 0; u < 3; u++)
#pragma unroll
      for (int w = 0; w < 3; w++) cd[u][w] = code[i + (ptrdiff_t)(u - 1) * p.pitch + (w - 1)];
    oo = oh_o[i];
#pragma unroll
    for (int k = 0; k < C; k++) {
      mc[k] = mu[idx(p, k, x, y)];
      mf[k] = mu[idx(p, k, x + 1, y)];
      mb[k] = mu[idx(p, k, x - 1, y)];
      mr[k] = mu[idx(p, k, x, y + 1)];
      ml[k] = mu[idx(p, k, x, y - 1)];
      lo[k] = Ops<R>::Exact ? R(0) : mulo[idx(p, k, x, y)];
    }
    cc = cd[1][1];
#pragma unroll
    for (int u = 0; u < 3; u++)
#pragma unroll
      for (int w = 0; w < 3; w++) cc = cd[u][w] == cc ? cc : -1;
    return cc < 0;
  }
  __device__ __forceinline__ void finish(const DevParams<R>& p, int x, int y, const R* __restrict__ mulo,
                                         R* __restrict__ phi_o, R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                         signed char* __restrict__ oh_o, R tb, int tsh) const {
    if (cc < 0) return;
    const R T = NI ? temp_row(p, tb, y, true, tsh) : R(0);
    // the bulk branch reads phase cc alone: one local phase (over all nine it
    // took 242 registers, or 552 B of scratch at six waves per SIMD; now 42)
    bulk_mu_onehot<C, R, NI>(p, cc, mc, mf, mb, mr, ml, mulo, mu_o, mulo_o, x, y, T, lo);
    if (oo != cc) {  // the same bits as ph + 0
#pragma unroll
      for (int a = 0; a < P; a++)
        write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, a == cc ? R(1.0) : R(0));
      oh_o[(size_t)x * p.pitch + y] = (signed char)cc;
    }
  }
};

// Light mu sweep of path 6 for the block whose cells are (x, y): the loads,
// the updates, and the cells left to the dense sweep appended to segment L &
// 7 of the mu-sweep list.  (Reserving the block's slots before the arithmetic,
// so that the atomic overlaps it, kept more registers live across the barrier
// and was not faster.)
template <int P, int C, class R, bool NI>
__device__ __forceinline__ void light_mu_block(const DevParams<R>& p, int x, int y, int L, int nblk,
                                               const R* __restrict__ mu, const R* __restrict__ mulo,
                                               const signed char* __restrict__ code, R* __restrict__ phi_o,
                                               R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                               signed char* __restrict__ oh_o, int* __restrict__ lc,
                                               int* __restrict__ cnt_c, R tb, int tsh) {
  LightMu<P, C, R, NI> lm;
  const bool in = x <= p.mesh_x + 2 && y <= p.mesh_y + 2;
  const bool heavy = in && lm.load(p, x, y, mu, mulo, code, oh_o);
  if (in) lm.finish(p, x, y, mulo, phi_o, mu_o, mulo_o, oh_o, tb, tsh);
  cell_append_seg<kMuCells>(heavy, x, y, L, nblk, lc, cnt_c);
}

// Dense phase sweep of path 6 over the segmented phase-sweep list (written by
// k_phase_light_oh's nbp blocks): phase_cell on listed cell i, i = first,
// first + stride, ...
template <int P, int C, class R, bool NI>
__device__ __forceinline__ void phase_cells_seg(const DevParams<R>& p, const R* __restrict__ phi,
                                                const R* __restrict__ mu, R* __restrict__ dphi,
                                                const int* __restrict__ lists, int nbp, int first, int stride, R tb,
                                                int tmode, const NoiseRef& nz) {
  const int* lp = lists + kSegInts;
  const SegList<kPhaseCells> sl(lists, nbp);
  for (int i = first; i < sl.n; i += stride) {
    const int e = lp[sl.seg_at(i)], x = e >> 16, y = e & 0xffff;
    if (x < 2 || x > p.rx - 3 || y < 2 || y > p.ry - 3) continue;  // entries are cells of the phase sweep
    phase_cell<P, C, R, NI>(p, phi, mu, dphi, x, y, NI ? temp_row(p, tb, y, (tmode & 1) != 0, tmode >> 1) : R(0), nz);
  }
}

// Dense phase sweep and light mu sweep of path 6 in one launch of BX x BY
// lanes per block.  Blocks [0, nd) take the phase-sweep list (phase_cells_seg);
// the gx x gy blocks after them (in the XCD-aware order of blk_xy; nd is a
// multiple of 8, so block L of them still goes to XCD L mod 8) sweep the
// interior (light_mu_block) and append the cells they leave to the segmented
// mu-sweep list (lists + kSegInts + capp, counters lists[kSegs kSegStride ..]).
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) __attribute__((amdgpu_waves_per_eu(GP_ONEHOT_WAVES)))
    k_phase_conc_oh(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi, const R* __restrict__ mu,
                    const R* __restrict__ mulo, R* __restrict__ dphi, const signed char* __restrict__ code,
                    R* __restrict__ phi_o, R* __restrict__ mu_o, R* __restrict__ mulo_o,
                    signed char* __restrict__ oh_o, int* __restrict__ lists, int nbp, int capp, int nd, int gx, R tb,
                    int tmode, int tsh, NoiseRef nz) {
  const DevParams<R>& p = *prm;
  if ((int)blockIdx.x < nd) {
    phase_cells_seg<P, C, R, NI>(p, phi, mu, dphi, lists, nbp, blockIdx.x * (BX * BY) + threadIdx.y * BX + threadIdx.x,
                                 nd * (BX * BY), tb, tmode, nz);
    return;
  }
  const int L = blockIdx.x - nd, n = gridDim.x - nd;
  const int q = n >> 3, r = n & 7, xcd = L & 7, s = L >> 3;
  const int l = xcd * q + min(xcd, r) + s;
  light_mu_block<P, C, R, NI>(p, 3 + (l / gx) * BY + threadIdx.y, 3 + (l % gx) * BX + threadIdx.x, L, n, mu, mulo, code,
                              phi_o, mu_o, mulo_o, oh_o, lists + kSegInts + capp, lists + kSegs * kSegStride, tb, tsh);
}

// The two halves of k_phase_conc_oh as launches of their own (each with its
// own register budget): the dense phase sweep on a 1-D grid of 256-lane
// blocks, then the light mu sweep on the gx x gy grid.  The one-hot path uses
// them where onehot_wide holds.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(onehot_dense_waves<P, R>()))) k_phase_cells_oh(const DevParams<R>* __restrict__ prm,
                                                                 const R* __restrict__ phi, const R* __restrict__ mu,
                                                                 R* __restrict__ dphi, const int* __restrict__ lists,
                                                                 int nbp, R tb, int tmode, NoiseRef nz) {
  phase_cells_seg<P, C, R, NI>(*prm, phi, mu, dphi, lists, nbp, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256, tb,
                               tmode, nz);
}

template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) k_conc_light_oh(const DevParams<R>* __restrict__ prm,
                                                           const R* __restrict__ mu, const R* __restrict__ mulo,
                                                           const signed char* __restrict__ code, R* __restrict__ phi_o,
                                                           R* __restrict__ mu_o, R* __restrict__ mulo_o,
                                                           signed char* __restrict__ oh_o, int* __restrict__ lists,
                                                           int capp, R tb, int tsh) {
  int bx, by;
  blk_xy(bx, by);
  light_mu_block<P, C, R, NI>(*prm, 3 + by * BY + threadIdx.y, 3 + bx * BX + threadIdx.x,
                              blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y, mu, mulo, code, phi_o, mu_o,
                              mulo_o, oh_o, lists + kSegInts + capp, lists + kSegs * kSegStride, tb, tsh);
}

// Dense mu sweep of path 6: the update of conc_cell_dense, with the new
// one-hot codes into oh_o, on the cells of the segmented mu-sweep list
// (written by the nbc light blocks of the mu sweep); one lane per cell where
// onehot_conc_one_lane holds, else two waves per cell: a
// block takes 128 listed cells per pass; waves 0-1 evaluate the x faces and
// finish the update, waves 2-3 evaluate the y faces of the same cells and hand
// them over in LDS.  One lane per cell left the kernel bound by the chain of
// one cell's arithmetic at one wave per SIMD; the halves' branches are uniform
// per wave, and each face is the same function of the same operands as in
// conc_cell_dense, so the bits are unchanged.  Clears the phase-sweep
// counters, whose readers have finished.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(onehot_dense_waves<P, R>()))) k_conc_cells_oh(const DevParams<R>* __restrict__ prm,
                                                                const R* __restrict__ phi, const R* __restrict__ mu,
                                                                const R* __restrict__ dphi,
                                                                const R* __restrict__ mulo, R* __restrict__ phi_o,
                                                                R* __restrict__ mu_o, R* __restrict__ mulo_o, R tb,
                                                                int tsh, int* __restrict__ lists, int capp, int nbc,
                                                                const signed char* __restrict__ code,
                                                                signed char* __restrict__ oh_o) {
  __shared__ R xch[128][2][C];
  const DevParams<R>& p = *prm;
  const int* lc = lists + kSegInts + capp;
  const SegList<kMuCells> sl(lists + kSegs * kSegStride, nbc);
  if (blockIdx.x == 0 && threadIdx.x < kSegs) lists[kSegStride * threadIdx.x] = 0;
  if constexpr (onehot_conc_one_lane<P, R>()) {  // one lane per listed cell
    for (int i = blockIdx.x * 256 + threadIdx.x; i < sl.n; i += gridDim.x * 256) {
      const int e = lc[sl.seg_at(i)], x = e >> 16, y = e & 0xffff;
      if (x < 3 || x > p.mesh_x + 2 || y < 3 || y > p.mesh_y + 2) continue;  // entries are interior cells
      conc_cell_dense<P, C, R, NI>(p, phi, mu, dphi, mulo, phi_o, mu_o, mulo_o, tb, tsh, code, oh_o, x, y);
    }
    return;
  }
  const int w = threadIdx.x >> 6, half = w >> 1, slot = (w & 1) * 64 + (threadIdx.x & 63);
  for (int base = blockIdx.x * 128; base < sl.n; base += gridDim.x * 128) {  // the same passes for every wave
    const int i = base + slot;
    int x = 0, y = 0;
    bool valid = i < sl.n;
    if (valid) {
      const int e = lc[sl.seg_at(i)];
      x = e >> 16;
      y = e & 0xffff;
      valid = x >= 3 && x <= p.mesh_x + 2 && y >= 3 && y <= p.mesh_y + 2;  // entries are interior cells
    }
    R v[P][3][3], dc[P], mc[C], mf[C], mb[C], mr[C], ml[C], ja[C], jz[C], Tc = R(0);
    if (valid) {
      Tc = NI ? temp_row(p, tb, y, true, tsh) : R(0);
      load3x3<P>(p, phi, x, y, v);
      Nbhd<P, R> nb;
      make_nbhd<P>(p, v, nb);
      R phc[P], pha[P], phz[P], da[P], dz[P];
#pragma unroll
      for (int a = 0; a < P; a++) phc[a] = v[a][1][1];
      load_dphi<P>(p, dphi, code, x, y, dc);
#pragma unroll
      for (int k = 0; k < C; k++) mc[k] = mu[idx(p, k, x, y)];
      if (half == 0) {  // +x and -x faces
#pragma unroll
        for (int a = 0; a < P; a++) {
          pha[a] = v[a][2][1];
          phz[a] = v[a][0][1];
        }
        load_dphi<P>(p, dphi, code, x + 1, y, da);
        load_dphi<P>(p, dphi, code, x - 1, y, dz);
#pragma unroll
        for (int k = 0; k < C; k++) {
          mf[k] = mu[idx(p, k, x + 1, y)];
          mb[k] = mu[idx(p, k, x - 1, y)];
          mr[k] = mu[idx(p, k, x, y + 1)];
          ml[k] = mu[idx(p, k, x, y - 1)];
        }
        face_jat<P, C, R, NI>(p, nb.gXc, nb.cYc, nb.cYf, phc, pha, mc, mf, dc, da, true, ja, Tc, Tc);
        face_jat<P, C, R, NI>(p, nb.gXb, nb.cYb, nb.cYc, phz, phc, mb, mc, dz, dc, true, jz, Tc, Tc);
      } else {  // +y and -y faces
        const R Tr = NI ? temp_row(p, tb, y + 1, true, tsh) : R(0);
        const R Tl = NI ? temp_row(p, tb, y - 1, true, tsh) : R(0);
#pragma unroll
        for (int a = 0; a < P; a++) {
          pha[a] = v[a][1][2];
          phz[a] = v[a][1][0];
        }
        load_dphi<P>(p, dphi, code, x, y + 1, da);
        load_dphi<P>(p, dphi, code, x, y - 1, dz);
#pragma unroll
        for (int k = 0; k < C; k++) {
          mr[k] = mu[idx(p, k, x, y + 1)];
          ml[k] = mu[idx(p, k, x, y - 1)];
        }
        face_jat<P, C, R, NI>(p, nb.gYc, nb.cXc, nb.cXr, phc, pha, mc, mr, dc, da, y != p.yskip, ja, Tc, Tr);
        face_jat<P, C, R, NI>(p, nb.gYl, nb.cXl, nb.cXc, phz, phc, ml, mc, dz, dc, (y - 1) != p.yskip, jz, Tl, Tc);
#pragma unroll
        for (int k = 0; k < C; k++) {
          xch[slot][0][k] = ja[k];
          xch[slot][1][k] = jz[k];
        }
      }
    }
    __syncthreads();
    if (valid && half == 0) {
      R jr[C], jl[C];
#pragma unroll
      for (int k = 0; k < C; k++) {
        jr[k] = xch[slot][0][k];
        jl[k] = xch[slot][1][k];
      }
      conc_apply<P, C, R, !Ops<R>::Exact, NI>(p, v, mc, mf, mb, mr, ml, dc, ja, jz, jr, jl, mulo, phi_o, mu_o, mulo_o,
                                             x, y, Tc);
      R pn[P];  // the exact one-hot code of the new phi (phc + dc, the value written)
#pragma unroll
      for (int a = 0; a < P; a++) pn[a] = v[a][1][1] + dc[a];
      oh_o[(size_t)x * p.pitch + y] = (signed char)onehot_bits<P>(pn);
    }
    __syncthreads();  // the exchange slots are refilled in the next pass
  }
}

// Sparse two-pass engine for interface tiles.  k_phase_tiles computes
// delta-phi on each listed tile plus its 1-cell ring into the dphi planes;
// k_conc_tiles then updates the tile.  Both kernels first sort the tile's cells
// in LDS into a cheap class (phase sweep: no active phase, projection only;
// concentration sweep: bulk_cell) handled at once and a list of full cells that
// the block's threads then share, so the expensive interface arithmetic runs on
// densely packed waves.
//
// The phase sweep also writes a one-byte code per cell: the phase a if phi is
// the exact one-hot vector of a and delta-phi is +0 in every phase, else -1.  A cell whose 3x3
// block carries one code a >= 0 meets the bulk_cell conditions.
template <int P, int C, class R, int TX, int TY>
__global__ void __launch_bounds__(256) GP_HEAVY k_phase_tiles(const Inst<R>* __restrict__ inst, const int* __restrict__ tinst,
                                                              int par, const int* __restrict__ list,
                                                              const int* __restrict__ count, int cap) {
  constexpr int RX1 = TX + 2, RY1 = TY + 2;
  __shared__ short todo[RX1 * RY1];
  __shared__ int ntodo;
  const int ntile = min(*count, cap);  // a list holds every tile at most once
  for (int it = blockIdx.x; it < ntile; it += gridDim.x) {
    const int tile = list[it];
    const Inst<R>& g = inst_of(inst, tinst, tile);
    const DevParams<R>& p = *g.prm;
    const R *phi = g.phi[par], *mu = g.mu[par];
    R* dphi = g.dphi;
    signed char* code = g.code;
    const int lt = tile - g.tile0;
    const int x0 = 3 + (lt / g.nty) * TX - 1, y0 = 3 + (lt % g.nty) * TY - 1;
    if (threadIdx.x == 0) ntodo = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < RX1 * RY1; i += 256) {
      const int x = x0 + i / RY1, y = y0 + i % RY1;
      if (x > p.rx - 3 || y > p.ry - 3) continue;
      R ph[P];
      if (phase_active<P>(p, phi, x, y, ph)) {
        todo[atomicAdd(&ntodo, 1)] = (short)i;
      } else {
        R dp[P];
        bool act[P];
#pragma unroll
        for (int a = 0; a < P; a++) {
          dp[a] = R(0);
          act[a] = false;
        }
        project_simplex<P>(ph, act, dp);
        bool zero = true;
#pragma unroll
        for (int a = 0; a < P; a++) {
          dphi[idx(p, a, x, y)] = dp[a];
          zero = zero && dp[a] == R(0) && !signbit(dp[a]);
        }
        code[(size_t)x * p.pitch + y] = (signed char)(zero ? onehot_bits<P>(ph) : -1);
        continue;
      }
      code[(size_t)x * p.pitch + y] = -1;
    }
    __syncthreads();
    const int n = ntodo;
    for (int j = threadIdx.x; j < n; j += 256) {
      const int i = todo[j];
      phase_cell<P, C>(p, phi, mu, dphi, x0 + i / RY1, y0 + i % RY1);
    }
    __syncthreads();
  }
}

template <int P, int C, class R, int TX, int TY>
__global__ void __launch_bounds__(256) GP_HEAVY k_conc_tiles(const Inst<R>* __restrict__ inst, const int* __restrict__ tinst,
                                                             int par, const int* __restrict__ list,
                                                             const int* __restrict__ count, int* __restrict__ flag_o,
                                                             int cap) {
  __shared__ int red[256];
  __shared__ short todo[TX * TY];
  __shared__ int ntodo;
  const int ntile = min(*count, cap);  // a list holds every tile at most once
  for (int it = blockIdx.x; it < ntile; it += gridDim.x) {
    const int tile = list[it];
    const Inst<R>& g = inst_of(inst, tinst, tile);
    const DevParams<R>& p = *g.prm;
    const R *phi = g.phi[par], *mu = g.mu[par], *mulo = g.mulo[par], *dphi = g.dphi;
    const signed char* code = g.code;
    R *phi_o = g.phi[par ^ 1], *mu_o = g.mu[par ^ 1], *mulo_o = g.mulo[par ^ 1];
    const int lt = tile - g.tile0;
    const int x0 = 3 + (lt / g.nty) * TX, y0 = 3 + (lt % g.nty) * TY;
    if (threadIdx.x == 0) ntodo = 0;
    __syncthreads();
    int f = -2;
    for (int i = threadIdx.x; i < TX * TY; i += 256) {
      const int x = x0 + i / TY, y = y0 + i % TY;
      if (x > p.mesh_x + 2 || y > p.mesh_y + 2) continue;
      int cc = code[(size_t)x * p.pitch + y];
#pragma unroll
      for (int u = -1; u <= 1; u++)
#pragma unroll
        for (int w = -1; w <= 1; w++) cc = code[(size_t)(x + u) * p.pitch + y + w] == cc ? cc : -1;
      if (cc >= 0) {
        bulk_cell<P, C, R>(p, phi, mu, mulo, phi_o, mu_o, mulo_o, x, y);
        f = flag_combine(f, cc);
      } else {
        todo[atomicAdd(&ntodo, 1)] = (short)i;
      }
    }
    __syncthreads();
    const int n = ntodo;
    for (int j = threadIdx.x; j < n; j += 256) {
      const int i = todo[j];
      f = flag_combine(f, conc_cell<P, C, R, !Ops<R>::Exact>(p, phi, mu, dphi, mulo, phi_o, mu_o, mulo_o,
                                                             x0 + i / TY, y0 + i % TY));
    }
    f = block_flag(f, red);
    if (threadIdx.x == 0) flag_o[tile] = f == -2 ? -1 : f;
  }
}

// Tile classification for one step: a tile is bulk when it and every tile its
// 2-cell halo reads from (deps, through the ghost copies) carry the same one-hot
// flag.  Appends to the interface / bulk lists with atomics on cnt[0..1] and
// clears the counters of the next step (cnt_next).
template <int Unused = 0>
__global__ void k_plan(const int* __restrict__ flag, const int* __restrict__ deps, int maxdep, int ntiles,
                       int* __restrict__ list_if, int* __restrict__ list_bulk, int* __restrict__ cnt,
                       int* __restrict__ cnt_next) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) {
    cnt_next[0] = 0;
    cnt_next[1] = 0;
  }
  const bool valid = t < ntiles;
  bool bulk = false;
  if (valid) {
    const int* d = deps + (size_t)t * (maxdep + 1);
    int f = flag[t], nd = d[0];
    bulk = f >= 0 && nd >= 0;
    for (int j = 1; bulk && j <= nd; j++) bulk = flag[d[j]] == f;
  }
  // one atomic per wave and list: lanes take consecutive slots
  const unsigned long long mb = __ballot(valid && bulk), mi = __ballot(valid && !bulk);
  const int lane = threadIdx.x & 63;
  int bb = 0, bi = 0;
  if (lane == 0) {
    if (mb) bb = atomicAdd(&cnt[1], __popcll(mb));
    if (mi) bi = atomicAdd(&cnt[0], __popcll(mi));
  }
  bb = __shfl(bb, 0);
  bi = __shfl(bi, 0);
  const unsigned long long below = (1ull << lane) - 1ull;
  if (valid) {
    // counters start at zero each step, so slots stay below ntiles; the tests
    // keep a stale counter from writing past the lists
    const int sb = bb + __popcll(mb & below), si = bi + __popcll(mi & below);
    if (bulk) {
      if (sb < ntiles) list_bulk[sb] = t;
    } else if (si < ntiles) {
      list_if[si] = t;
    }
  }
}

// Clears both counter pairs of the sparse steps (a kernel, not a memset node,
// so that it may sit in a captured graph).
template <int Unused = 0>
__global__ void k_clear_counts(int* __restrict__ cnt) {
  if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
}

// Whether every phi ghost image of interior cell (x, y) holds the exact one-hot
// vector of phase f.  After a frame shift the ghost layers are not images: the
// rows were moved as they lay, and no boundary copy followed.
template <int P, class R>
__device__ __forceinline__ bool ghosts_hold(const DevParams<R>& p, const R* __restrict__ phi, int x, int y, int f) {
  if (x >= p.gfree[0][0][0] && x <= p.gfree[0][0][1] && y >= p.gfree[0][1][0] && y <= p.gfree[0][1][1]) return true;
  bool held = true;
#pragma unroll 1
  for (int i = -1; i < 6; i++) {  // x itself, then its images
    if (i >= 0 && p.gsrc[0][0][i] != x) continue;
    const int gx = i < 0 ? x : ghost_index(i, p.rx);
#pragma unroll 1
    for (int j = -1; j < 6; j++) {
      if (j >= 0 && p.gsrc[0][1][j] != y) continue;
      const int gy = j < 0 ? y : ghost_index(j, p.ry);
      R ph[P];
#pragma unroll
      for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, gx, gy)];
      held = held && onehot_bits<P>(ph) == f;
    }
  }
  return held;
}

// Flags of a state that no step of the tile paths left (one block per tile);
// those of the other buffer, of unknown contents, are cleared.  A flag vouches
// for the tile's cells and for their ghost images: k_plan takes a ghost cell for
// its source, and k_bulk leaves both unwritten where the flag is the phase it
// would write.  A tile whose images differ is an interface tile for one step,
// which reads the ghost layers as they are.
template <int P, class R, int TX, int TY>
__global__ void __launch_bounds__(256) k_flags(const Inst<R>* __restrict__ inst, const int* __restrict__ tinst,
                                               int par, int* __restrict__ flag, int* __restrict__ flag_x) {
  __shared__ int red[256];
  const int tile = blockIdx.x;
  const Inst<R>& g = inst_of(inst, tinst, tile);
  const DevParams<R>& p = *g.prm;
  const R* phi = g.phi[par];
  const int lt = tile - g.tile0;
  const int x0 = 3 + (lt / g.nty) * TX, y0 = 3 + (lt % g.nty) * TY;
  int f = -2;
  for (int i = threadIdx.x; i < TX * TY; i += 256) {
    const int x = x0 + i / TY, y = y0 + i % TY;
    if (x > p.mesh_x + 2 || y > p.mesh_y + 2) continue;
    R ph[P];
#pragma unroll
    for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, x, y)];
    const int cf = onehot_bits<P>(ph);
    f = flag_combine(f, cf >= 0 && !ghosts_hold<P>(p, phi, x, y, cf) ? -1 : cf);
  }
  f = block_flag(f, red);
  if (threadIdx.x == 0) {
    flag[tile] = f == -2 ? -1 : f;
    flag_x[tile] = -1;
  }
}

}  // namespace GPK_NS
