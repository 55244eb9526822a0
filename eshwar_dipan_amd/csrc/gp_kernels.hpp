// gp_kernels.hpp -- gfx950 kernels of the grand-potential 2-D step.
//
// Field storage: one plane per phase / component, rows_x = MESH_X+6 rows of
// `pitch` elements (y fastest, pitch >= MESH_Y+6 rounded to 256 bytes), i.e. the
// reference's padded grid with its three ghost layers (solverloop/serialinfo_xy.h:7-16).
//
// Two-pass path:
//   k_phase      : delta-phi on x,y in [2, rows-3] (interior plus the ghost ring
//                  the antitrapping fluxes read)        -- solverloop_phasefield
//   k_conc_lds / : mu and phi update of the interior, written out-of-place, each
//   k_conc_march   cell also written to the ghost cells that copy it (so the ghost
//                  copies of apply_boundary_conditions need no separate pass);
//                  antitrapping faces shared between cells -- solverloop_concentration
// Fused path (one launch per step): see k_fused in gp_fused.hpp.
#pragma once

#include <stdint.h>

#include "gp_cell.hpp"

// Waves per SIMD that the interface kernels are compiled for: their cell
// arithmetic holds a few hundred values live, and without a bound the compiler
// spends the whole register file on one wave per SIMD, which leaves the FP64
// and memory latencies unhidden.
#ifndef GP_WAVES_PER_EU
#define GP_WAVES_PER_EU 2
#endif
#define GP_HEAVY __attribute__((amdgpu_waves_per_eu(GP_WAVES_PER_EU)))
#ifndef GP_ONEHOT_WAVES
#define GP_ONEHOT_WAVES GP_WAVES_PER_EU  // the one-hot path's launch of its dense phase and light mu sweeps
#endif
#ifndef GP_CONC_WAVES
#define GP_CONC_WAVES GP_WAVES_PER_EU
#endif

namespace GPK_NS {

// At nine or more phases the one-hot path runs its dense phase sweep as a
// launch of its own, so that the light mu sweep is not held to the dense
// sweep's register budget (4096^2, 9 phases, binary32: 1.49e10 -> 1.64e10
// cell-updates/s).  Binary64 there needs more registers than two waves per
// SIMD leave (the dense phase sweep spilled 2.5 KB per lane, the dense mu
// sweep 0.6 KB): its dense sweeps run at one wave per SIMD (1.6x the merged
// launch at two waves).  Binary32 spills 0.8 KB and is faster at two waves.
template <int P, class R>
constexpr bool onehot_wide() { return P >= 9; }
template <int P, class R>
constexpr int onehot_dense_waves() { return onehot_wide<P, R>() && sizeof(R) == 8 ? 1 : GP_WAVES_PER_EU; }
// The one-hot path's dense mu sweep takes two waves per listed cell (the x and
// y antitrapping faces side by side) below nine phases, one lane per cell from
// nine: at 4096^2 and nine phases one lane is 15% (binary64) and 6% (binary32)
// faster, at 1024^2 and four phases two waves are faster.
template <int P, class R>
constexpr bool onehot_conc_one_lane() { return P >= 9; }

constexpr int BX = 64;  // threads along y (contiguous)
constexpr int BY = 4;   // threads along x

// XCD-aware block order.  Workgroups are dispatched to the 8 XCDs round-robin
// by linear id, and each XCD has its own L2, so with the natural order the
// stencil halo rows between neighbouring blocks are fetched into different
// L2s.  blk_xy maps the linear id L (XCD L % 8, its (L / 8)-th block) to a
// logical block of a contiguous range per XCD, in dispatch order, so that an
// XCD sweeps its own band of rows and its L2 holds the halo it re-reads.  The
// map is a bijection of [0, gridDim.x * gridDim.y).
__device__ __forceinline__ void blk_xy(int& bx, int& by) {
  const int n = gridDim.x * gridDim.y, L = blockIdx.y * gridDim.x + blockIdx.x;
  const int q = n >> 3, r = n & 7, xcd = L & 7, s = L >> 3;
  const int l = xcd * q + min(xcd, r) + s;
  bx = l % gridDim.x;
  by = l / gridDim.x;
}

// Block of a list-driven launch (split two-pass step): block i of a 1-D grid
// takes logical block list[i] of a gx-wide grid; blocks past *count return.
// Without a list, the XCD-aware order of the full 2-D grid.
__device__ __forceinline__ bool blk_pick(const int* __restrict__ list, const int* __restrict__ count, int gx, int& bx,
                                         int& by) {
  if (!list) {
    blk_xy(bx, by);
    return true;
  }
  if ((int)blockIdx.x >= min(*count, (int)gridDim.x)) return false;  // the 1-D grid spans every block
  const int l = list[blockIdx.x];
  bx = l % gx;
  by = l / gx;
  return true;
}

// Phase-field noise of one step (gp_noise.hpp), all device memory; raw ==
// nullptr: no noise.
struct NoiseRef {
  const uint32_t* raw;  // the step's glibc rand() words, in draw order
  const int* cell_off;  // [x][y] (plane layout): draws before (x, y) in its row
  const int* row_base;  // [x]: draws before row x
  double amp;           // Amp_Noise_Phase
};

template <class R>
__device__ __forceinline__ size_t idx(const DevParams<R>& p, int a, int x, int y) {
  return (size_t)a * p.plane + (size_t)x * p.pitch + y;
}

// Padded ghost indices of slot s (0..5) along an axis of n padded rows.
__device__ __forceinline__ int ghost_index(int s, int n) { return s < 3 ? s : n - 6 + s; }

// Write value v of field plane `base` at interior (x,y) and at every ghost cell
// whose copy source is (x,y) for field f (X faces first then Y faces in the
// reference, so a corner ghost holds the value at (proxy_x, proxy_y)).
template <class R>
__device__ __forceinline__ void write_with_ghosts(const DevParams<R>& p, int f, R* __restrict__ base, int x, int y, R v) {
  if (x >= p.gfree[f][0][0] && x <= p.gfree[f][0][1] && y >= p.gfree[f][1][0] && y <= p.gfree[f][1][1]) {
    base[(size_t)x * p.pitch + y] = v;  // the source of no ghost image
    return;
  }
  int tx[3], ty[3], nx = 1, ny = 1;
  tx[0] = x;
  ty[0] = y;
#pragma unroll
  for (int s = 0; s < 6; s++) {
    if (p.gsrc[f][0][s] == x) tx[nx++] = ghost_index(s, p.rx);
    if (p.gsrc[f][1][s] == y) ty[ny++] = ghost_index(s, p.ry);
  }
  for (int i = 0; i < nx; i++)
    for (int j = 0; j < ny; j++) base[(size_t)tx[i] * p.pitch + ty[j]] = v;
}

// Delta-phi of cell (x, y).  Given the split path's codes, a cell with code
// >= 0 has delta-phi +0 in every phase (the code is written only then), and
// the light phase sweep leaves its planes unwritten.
template <int P, class R>
__device__ __forceinline__ void load_dphi(const DevParams<R>& p, const R* __restrict__ dphi,
                                          const signed char* __restrict__ code, int x, int y, R (&d)[P]) {
  if (code && code[(size_t)x * p.pitch + y] >= 0) {
#pragma unroll
    for (int a = 0; a < P; a++) d[a] = R(0);
  } else {
#pragma unroll
    for (int a = 0; a < P; a++) d[a] = dphi[idx(p, a, x, y)];
  }
}

template <int P, class R>
__device__ __forceinline__ void load3x3(const DevParams<R>& p, const R* __restrict__ phi, int x, int y, R (&v)[P][3][3]) {
#pragma unroll
  for (int a = 0; a < P; a++)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) v[a][i][j] = phi[idx(p, a, x + i - 1, y + j - 1)];
}

// delta-phi of padded cell (x,y) into dphi (calculate_divergence_phasefield_2D)
template <int P, int C, class R, bool NI = false>
__device__ __forceinline__ void phase_cell(const DevParams<R>& p, const R* __restrict__ phi, const R* __restrict__ mu,
                                           R* __restrict__ dphi, int x, int y, R T = R(0),
                                           const NoiseRef& nz = NoiseRef{}) {
  R v[P][3][3];
  load3x3<P>(p, phi, x, y, v);
  Nbhd<P, R> n;
  make_nbhd<P>(p, v, n);
  R m[C], dp[P];
#pragma unroll
  for (int k = 0; k < C; k++) m[k] = mu[idx(p, k, x, y)];
  const uint32_t* nzw = nz.raw ? nz.raw + nz.row_base[x] + nz.cell_off[(size_t)x * p.pitch + y] : nullptr;
  cell_dphi<P, C, R, NI>(p, n, m, dp, T, nzw, (R)nz.amp);
#pragma unroll
  for (int a = 0; a < P; a++) dphi[idx(p, a, x, y)] = dp[a];
}

// mu and phi update of interior cell (x,y) from its 3x3 phi block v, the mu of
// its five-point stencil, its delta-phi and the antitrapping fluxes of its four
// faces; writes the cell and its ghost images.  Kahan adds the mu increment to
// mu + mulo (binary32).  Returns the phase of which the updated phi is
// the exact one-hot vector (-1 if none).
template <int P, int C, class R, bool Kahan, bool NI = false>
__device__ __forceinline__ int conc_apply(const DevParams<R>& p, const R (&v)[P][3][3], const R* mc, const R* mf,
                                          const R* mb, const R* mr, const R* ml, const R* dc, const R* jf,
                                          const R* jb, const R* jr, const R* jl, const R* __restrict__ mulo,
                                          R* __restrict__ phi_o, R* __restrict__ mu_o, R* __restrict__ mulo_o, int x,
                                          int y, R T = R(0), R* __restrict__ comp = nullptr) {
  R phc[P], phf[P], phb[P], phr[P], phl[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    phc[a] = v[a][1][1];
    phf[a] = v[a][2][1];
    phb[a] = v[a][0][1];
    phr[a] = v[a][1][2];
    phl[a] = v[a][1][0];
  }
  // face mobilities and mu gradients (calculate_gradients.h:148-165)
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
  if (comp) {  // composition field, updated in place (each cell reads only its own)
    R cst[C];
#pragma unroll
    for (int k = 0; k < C; k++) cst[k] = comp[idx(p, k, x, y)];
    cell_update<P, C, R, NI>(p, phc, mc, dc, jf, jb, jr, jl, Dmf, Dmb, Dmr, Dml, gmf, gmb, gmr, gml, pho, muo, dmu, T,
                             cst);
#pragma unroll
    for (int k = 0; k < C; k++) write_with_ghosts(p, 1, comp + (size_t)k * p.plane, x, y, cst[k]);
  } else {
    cell_update<P, C, R, NI>(p, phc, mc, dc, jf, jb, jr, jl, Dmf, Dmb, Dmr, Dml, gmf, gmb, gmr, gml, pho, muo, dmu, T);
  }
#pragma unroll
  for (int a = 0; a < P; a++) write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, pho[a]);
  if constexpr (!Kahan) {
#pragma unroll
    for (int k = 0; k < C; k++) write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, muo[k]);
  } else {
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
  int a1 = -1, n1 = 0, nz = 0;  // the exact one-hot bits
#pragma unroll
  for (int a = 0; a < P; a++) {
    if (pho[a] == R(1.0)) {
      a1 = a;
      n1++;
    } else if (pho[a] != R(0) || signbit(pho[a])) {
      nz++;
    }
  }
  return nz == 0 && n1 == 1 ? a1 : -1;
}

// mu and phi update of interior cell (x,y) with its ghost images (all four
// face fluxes computed here).  Returns the one-hot phase as conc_apply.
template <int P, int C, class R, bool Kahan>
__device__ __forceinline__ int conc_cell(const DevParams<R>& p, const R* __restrict__ phi, const R* __restrict__ mu,
                                         const R* __restrict__ dphi, const R* __restrict__ mulo, R* __restrict__ phi_o,
                                         R* __restrict__ mu_o, R* __restrict__ mulo_o, int x, int y,
                                         R* __restrict__ comp = nullptr) {
  R v[P][3][3];
  load3x3<P>(p, phi, x, y, v);
  Nbhd<P, R> n;
  make_nbhd<P>(p, v, n);
  R phc[P], phf[P], phb[P], phr[P], phl[P];
  R dc[P], df[P], db[P], dr[P], dl[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    phc[a] = v[a][1][1];
    phf[a] = v[a][2][1];
    phb[a] = v[a][0][1];
    phr[a] = v[a][1][2];
    phl[a] = v[a][1][0];
    dc[a] = dphi[idx(p, a, x, y)];
    df[a] = dphi[idx(p, a, x + 1, y)];
    db[a] = dphi[idx(p, a, x - 1, y)];
    dr[a] = dphi[idx(p, a, x, y + 1)];
    dl[a] = dphi[idx(p, a, x, y - 1)];
  }
  R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    mc[k] = mu[idx(p, k, x, y)];
    mf[k] = mu[idx(p, k, x + 1, y)];
    mb[k] = mu[idx(p, k, x - 1, y)];
    mr[k] = mu[idx(p, k, x, y + 1)];
    ml[k] = mu[idx(p, k, x, y - 1)];
  }
  // antitrapping on the four faces
  R jf[C], jb[C], jr[C], jl[C];
  face_jat<P, C>(p, n.gXc, n.cYc, n.cYf, phc, phf, mc, mf, dc, df, true, jf);
  face_jat<P, C>(p, n.gXb, n.cYb, n.cYc, phb, phc, mb, mc, db, dc, true, jb);
  face_jat<P, C>(p, n.gYc, n.cXc, n.cXr, phc, phr, mc, mr, dc, dr, y != p.yskip, jr);
  face_jat<P, C>(p, n.gYl, n.cXl, n.cXc, phl, phc, ml, mc, dl, dc, (y - 1) != p.yskip, jl);
  return conc_apply<P, C, R, Kahan>(p, v, mc, mf, mb, mr, ml, dc, jf, jb, jr, jl, mulo, phi_o, mu_o, mulo_o, x, y,
                                    R(0), comp);
}

// delta-phi on [2, rows-3]^2, one cell per thread
__host__ __device__ inline dim3 phase_grid(int rx, int ry) { return dim3((ry - 4 + BX - 1) / BX, (rx - 4 + BY - 1) / BY); }

// With NI (non-isothermal), tb is temp_bottom of this step; bit 0 of tmode tells
// whether the temperature ghost rows hold their boundary copies (first step
// after the copies) or the linear profile, and tmode >> 1 is the row shift of
// the step after a moving-frame shift (temp_row).
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) GP_HEAVY k_phase(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                   const R* __restrict__ mu, R* __restrict__ dphi, R tb = R(0),
                                                   int tmode = 0, const int* __restrict__ list = nullptr,
                                                   const int* __restrict__ count = nullptr, int gx = 0,
                                                   NoiseRef nz = NoiseRef{}) {
  const DevParams<R>& p = *prm;
  int bx, by;
  if (!blk_pick(list, count, gx, bx, by)) return;
  const int y = 2 + bx * BX + threadIdx.x;
  const int x = 2 + by * BY + threadIdx.y;
  if (x > p.rx - 3 || y > p.ry - 3) return;
  phase_cell<P, C, R, NI>(p, phi, mu, dphi, x, y, NI ? temp_row(p, tb, y, (tmode & 1) != 0, tmode >> 1) : R(0), nz);
}

// ---------------------------------------------------------------- MPI solver semantics
// Two-pass step with the F_01 semantics of the reference's MPI solver
// (gp_params.mpi), one cell per thread; binary64, isothermal.
//
// k_phase_mpi: delta-phi of padded cell (x, y) of [2, rows-3]^2 as
// phase_cell, with dpsi / V and the drand48 noise of the cell (one draw per
// cell of [1, rows-2]^2 in sweep order, x outer: draw (x-1)(rows_y-2) + y
// after the step's state).  With GP_MPI_GHOST_DPHI the ghost cells take their
// source's delta-phi (the boundary copies after the phase sweep copy it,
// MPI boundary_mpi.h:94-105): interior cells write it to their ghost images and
// ghost cells write nothing.
template <int P, int C, class R>
__global__ void __launch_bounds__(BX * BY) GP_HEAVY k_phase_mpi(const DevParams<R>* __restrict__ prm,
                                                                const R* __restrict__ phi, const R* __restrict__ mu,
                                                                R* __restrict__ dphi) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 2 + bx * BX + threadIdx.x;
  const int x = 2 + by * BY + threadIdx.y;
  if (x > p.rx - 3 || y > p.ry - 3) return;
  const bool ghost = x < 3 || x > p.mesh_x + 2 || y < 3 || y > p.mesh_y + 2;
  const bool copy = (p.mpi & GP_MPI_GHOST_DPHI) != 0;
  if (copy && ghost) return;
  R v[P][3][3];
  load3x3<P>(p, phi, x, y, v);
  Nbhd<P, R> n;
  make_nbhd<P>(p, v, n);
  R m[C], dp[P];
#pragma unroll
  for (int k = 0; k < C; k++) m[k] = mu[idx(p, k, x, y)];
  R mnz = R(0);
  if (p.mpi_noise) {
    const unsigned long long j = (unsigned long long)(x - 1) * (unsigned long long)(p.ry - 2) + (unsigned long long)y;
    mnz = p.noise4amp * (R)lcg_draw(p, *p.rstate, j);
  }
  cell_dphi<P, C, R, false, true>(p, n, m, dp, R(0), nullptr, R(0), mnz);
  if (copy) {
#pragma unroll
    for (int a = 0; a < P; a++) write_with_ghosts(p, 0, dphi + (size_t)a * p.plane, x, y, dp[a]);
  } else {
#pragma unroll
    for (int a = 0; a < P; a++) dphi[idx(p, a, x, y)] = dp[a];
  }
}

// The drand48 state after one step's draws (one thread).
template <class R>
__global__ void k_lcg_advance(const DevParams<R>* __restrict__ prm) {
  const DevParams<R>& p = *prm;
  if (threadIdx.x == 0 && blockIdx.x == 0) *p.rstate = (p.lcg_step[0] * *p.rstate + p.lcg_step[1]) & kLcgMask;
}

// k_conc_mpi: mu and phi update of interior cell (x, y), its four faces
// evaluated by its own thread (conc_cell), with the composition field when
// p.comp is set.
template <int P, int C, class R>
__global__ void __launch_bounds__(BX * BY) GP_HEAVY k_conc_mpi(const DevParams<R>* __restrict__ prm,
                                                               const R* __restrict__ phi, const R* __restrict__ mu,
                                                               const R* __restrict__ dphi, R* __restrict__ phi_o,
                                                               R* __restrict__ mu_o) {
  const DevParams<R>& p = *prm;
  int bx, by;
  blk_xy(bx, by);
  const int y = 3 + bx * BX + threadIdx.x;
  const int x = 3 + by * BY + threadIdx.y;
  if (x > p.mesh_x + 2 || y > p.mesh_y + 2) return;
  conc_cell<P, C, R, false>(p, phi, mu, dphi, nullptr, phi_o, mu_o, nullptr, x, y, p.comp);
}

// Composition of every interior cell from the fields, c_k = sum_a h_a(phi)
// c_a,k(mu), with its ghost images (the initial composition of a state given
// as phi and mu).
template <int P, int C, class R>
__global__ void k_comp_init(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi, const R* __restrict__ mu) {
  const DevParams<R>& p = *prm;
  const int y = 3 + blockIdx.x * blockDim.x + threadIdx.x;
  const int x = 3 + blockIdx.y;
  if (x > p.mesh_x + 2 || y > p.mesh_y + 2) return;
  R ph[P], m[C];
#pragma unroll
  for (int a = 0; a < P; a++) ph[a] = phi[idx(p, a, x, y)];
#pragma unroll
  for (int k = 0; k < C; k++) m[k] = mu[idx(p, k, x, y)];
#pragma unroll
  for (int k = 0; k < C; k++) {
    R c = R(0);
#pragma unroll
    for (int a = 0; a < P; a++) c += hphi<P>(ph, a) * c_mu<C>(p, m, a, k);
    write_with_ghosts(p, 1, p.comp + (size_t)k * p.plane, x, y, c);
  }
}

// mu and phi update of the interior with shared faces.  The antitrapping flux of a face is the same
// function of the same operands whichever of its two cells evaluates it
// (face_jat on the pair (lower, upper)), so a face need not be evaluated
// twice: a wave holds 64 consecutive y columns, starting one column before the
// 63 cells it updates, and marches KM rows along x.  Each lane evaluates the
// +x and +y faces of its cell; the -y flux comes from the lane below, the -x
// flux of row i > 0 is the +x flux of row i-1 and the first row evaluates its
// own.  That is 1 + 1/KM + 64/63 face evaluations per cell instead of 4.
// KM = 1 is the fastest at 1024^2 with four phases (on 256 CUs more waves in
// flight outweigh the shared x faces; KM = 2, 3, 4 were 2.5%, 4% and 8.5%
// slower in binary64).  Lanes past the last column read a clamped column and
// write nothing.
#ifndef GP_KM
#define GP_KM 1
#endif
constexpr int KM = GP_KM;  // rows per wave
constexpr int MW = 63;    // cells per wave along y

template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) __attribute__((amdgpu_waves_per_eu(GP_CONC_WAVES))) k_conc_march(const DevParams<R>* __restrict__ prm,
                                                              const R* __restrict__ phi, const R* __restrict__ mu,
                                                              const R* __restrict__ dphi, const R* __restrict__ mulo,
                                                              R* __restrict__ phi_o, R* __restrict__ mu_o,
                                                              R* __restrict__ mulo_o, R tb = R(0), int tsh = 0,
                                                              const int* __restrict__ list = nullptr,
                                                              const int* __restrict__ count = nullptr, int gx = 0,
                                                              const signed char* __restrict__ code = nullptr) {
  const DevParams<R>& p = *prm;
  const int lane = threadIdx.x;
  int bx, by;
  if (!blk_pick(list, count, gx, bx, by)) return;
  const int y = 2 + bx * MW + lane;  // lane 0 sits one column before the wave's cells
  const int yc = min(y, p.mesh_y + 2);
  // temperatures of the cell row and of the row above (the sweep runs after the boundary copies)
  const R Tc = NI ? temp_row(p, tb, yc, true, tsh) : R(0), Tr = NI ? temp_row(p, tb, yc + 1, true, tsh) : R(0);
  const bool cell = lane > 0 && y <= p.mesh_y + 2;
  const int x0 = 3 + (by * BY + threadIdx.y) * KM;
  if (x0 > p.mesh_x + 2) return;  // uniform over the wave
  R v[P][3][3];
  load3x3<P>(p, phi, x0, yc, v);
  R dc[P], jb[C];
  load_dphi<P>(p, dphi, code, x0, yc, dc);
  {
    Nbhd<P, R> n;
    make_nbhd<P>(p, v, n);
    R phb[P], phc[P], db[P], mb[C], mc[C];
#pragma unroll
    for (int a = 0; a < P; a++) {
      phb[a] = v[a][0][1];
      phc[a] = v[a][1][1];
    }
    load_dphi<P>(p, dphi, code, x0 - 1, yc, db);
#pragma unroll
    for (int k = 0; k < C; k++) {
      mb[k] = mu[idx(p, k, x0 - 1, yc)];
      mc[k] = mu[idx(p, k, x0, yc)];
    }
    face_jat<P, C, R, NI>(p, n.gXb, n.cYb, n.cYc, phb, phc, mb, mc, db, dc, true, jb, Tc, Tc);
  }
  for (int i = 0; i < KM; i++) {
    const int x = x0 + i;
    if (x > p.mesh_x + 2) break;  // uniform over the wave
    if (i > 0) {
#pragma unroll
      for (int a = 0; a < P; a++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
          v[a][0][j] = v[a][1][j];
          v[a][1][j] = v[a][2][j];
          v[a][2][j] = phi[idx(p, a, x + 1, yc + j - 1)];
        }
    }
    Nbhd<P, R> n;
    make_nbhd<P>(p, v, n);
    R phc[P], phf[P], phr[P], df[P], dr[P];
#pragma unroll
    for (int a = 0; a < P; a++) {
      phc[a] = v[a][1][1];
      phf[a] = v[a][2][1];
      phr[a] = v[a][1][2];
    }
    load_dphi<P>(p, dphi, code, x + 1, yc, df);
    load_dphi<P>(p, dphi, code, x, yc + 1, dr);
    R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
    for (int k = 0; k < C; k++) {
      mc[k] = mu[idx(p, k, x, yc)];
      mf[k] = mu[idx(p, k, x + 1, yc)];
      mb[k] = mu[idx(p, k, x - 1, yc)];
      mr[k] = mu[idx(p, k, x, yc + 1)];
      ml[k] = mu[idx(p, k, x, yc - 1)];
    }
    R jf[C], jr[C], jl[C];
    face_jat<P, C, R, NI>(p, n.gXc, n.cYc, n.cYf, phc, phf, mc, mf, dc, df, true, jf, Tc, Tc);
    face_jat<P, C, R, NI>(p, n.gYc, n.cXc, n.cXr, phc, phr, mc, mr, dc, dr, yc != p.yskip, jr, Tc, Tr);
#pragma unroll
    for (int k = 0; k < C; k++) jl[k] = __shfl_up(jr[k], 1);
    if (cell)
      conc_apply<P, C, R, !Ops<R>::Exact, NI>(p, v, mc, mf, mb, mr, ml, dc, jf, jb, jr, jl, mulo, phi_o, mu_o, mulo_o, x, y, Tc);
#pragma unroll
    for (int k = 0; k < C; k++) jb[k] = jf[k];
#pragma unroll
    for (int a = 0; a < P; a++) dc[a] = df[a];
  }
}

// k_conc_march with KM = 1 and the x faces shared through LDS: the four waves
// of a block hold four consecutive x rows; each wave evaluates the +x and +y
// faces of its row, the first wave also its -x face, and the -x flux of row
// w > 0 is read from row w-1 after a barrier.  1 + 1/BY + 64/63 face
// evaluations per cell.
template <int P, int C, class R, bool NI = false>
__global__ void __launch_bounds__(BX * BY) __attribute__((amdgpu_waves_per_eu(GP_CONC_WAVES))) k_conc_lds(const DevParams<R>* __restrict__ prm,
                                                            const R* __restrict__ phi, const R* __restrict__ mu,
                                                            const R* __restrict__ dphi, const R* __restrict__ mulo,
                                                            R* __restrict__ phi_o, R* __restrict__ mu_o,
                                                            R* __restrict__ mulo_o, R tb = R(0), int tsh = 0,
                                                            const int* __restrict__ list = nullptr,
                                                            const int* __restrict__ count = nullptr, int gx = 0,
                                                            const signed char* __restrict__ code = nullptr) {
  __shared__ R jx[C][BY][BX];
  const DevParams<R>& p = *prm;
  const int lane = threadIdx.x, w = threadIdx.y;
  int bx, by;
  if (!blk_pick(list, count, gx, bx, by)) return;  // uniform over the block
  const int y = 2 + bx * MW + lane;  // lane 0 sits one column before the wave's cells
  const int yc = min(y, p.mesh_y + 2);
  // temperatures of the cell row and of the row above (the sweep runs after the boundary copies)
  const R Tc = NI ? temp_row(p, tb, yc, true, tsh) : R(0), Tr = NI ? temp_row(p, tb, yc + 1, true, tsh) : R(0);
  const int x = 3 + by * BY + w;
  const int xc = min(x, p.mesh_x + 2);       // waves past the last row compute a copy and write nothing
  const bool cell = x <= p.mesh_x + 2 && lane > 0 && y <= p.mesh_y + 2;
  R v[P][3][3];
  load3x3<P>(p, phi, xc, yc, v);
  Nbhd<P, R> n;
  make_nbhd<P>(p, v, n);
  R phc[P], phf[P], phr[P], dc[P], df[P], dr[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    phc[a] = v[a][1][1];
    phf[a] = v[a][2][1];
    phr[a] = v[a][1][2];
  }
  load_dphi<P>(p, dphi, code, xc, yc, dc);
  load_dphi<P>(p, dphi, code, xc + 1, yc, df);
  load_dphi<P>(p, dphi, code, xc, yc + 1, dr);
  R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    mc[k] = mu[idx(p, k, xc, yc)];
    mf[k] = mu[idx(p, k, xc + 1, yc)];
    mb[k] = mu[idx(p, k, xc - 1, yc)];
    mr[k] = mu[idx(p, k, xc, yc + 1)];
    ml[k] = mu[idx(p, k, xc, yc - 1)];
  }
  R jf[C], jb[C], jr[C], jl[C];
  face_jat<P, C, R, NI>(p, n.gXc, n.cYc, n.cYf, phc, phf, mc, mf, dc, df, true, jf, Tc, Tc);
  face_jat<P, C, R, NI>(p, n.gYc, n.cXc, n.cXr, phc, phr, mc, mr, dc, dr, yc != p.yskip, jr, Tc, Tr);
#pragma unroll
  for (int k = 0; k < C; k++) {
    jl[k] = __shfl_up(jr[k], 1);
    jx[k][w][lane] = jf[k];
  }
  if (w == 0) {  // uniform over the wave
    R phb[P], db[P];
#pragma unroll
    for (int a = 0; a < P; a++) phb[a] = v[a][0][1];
    load_dphi<P>(p, dphi, code, xc - 1, yc, db);
    face_jat<P, C, R, NI>(p, n.gXb, n.cYb, n.cYc, phb, phc, mb, mc, db, dc, true, jb, Tc, Tc);
  }
  __syncthreads();
  if (w > 0) {
#pragma unroll
    for (int k = 0; k < C; k++) jb[k] = jx[k][w - 1][lane];
  }
  if (cell)
    conc_apply<P, C, R, !Ops<R>::Exact, NI>(p, v, mc, mf, mb, mr, ml, dc, jf, jb, jr, jl, mulo, phi_o, mu_o, mulo_o, x, y, Tc);
}

// One two-pass step on `stream`: delta-phi of (phi, mu) into dphi, then the
// update into (phi_o, mu_o[, mulo_o]) with shared antitrapping faces.
// Binary64 shares x faces through LDS (3% faster at 1024^2, P=4); in binary32
// the barrier costs more than the face it saves (1% slower), so one row per
// wave.  The sharing kernels beat one cell per thread also at two phases
// (512^2: 1.3% in binary64, 5% in binary32; equal at 256^2).
// With NI (non-isothermal), tb is temp_bottom of the step, tproxy whether the
// phase sweep sees the temperature boundary copies (first step after them) and
// tsh the row shift of the step after a moving-frame shift.
template <int P, int C, class R, bool NI = false>
void launch_two_pass(const DevParams<R>* prm, int rx, int ry, int mesh_x, int mesh_y, hipStream_t stream,
                     const R* phi, const R* mu, R* dphi, const R* mulo, R* phi_o, R* mu_o, R* mulo_o,
                     R tb = R(0), int tproxy = 0, int tsh = 0, NoiseRef nz = NoiseRef{}) {
  const dim3 blk(BX, BY);
  hipLaunchKernelGGL((k_phase<P, C, R, NI>), phase_grid(rx, ry), blk, 0, stream, prm, phi, mu, dphi, tb,
                     (tproxy ? 1 : 0) | (tsh << 1), (const int*)nullptr, (const int*)nullptr, 0, nz);
  constexpr bool lds = Ops<R>::Exact;
  constexpr int rows = BY * (lds ? 1 : KM);
  const dim3 g((mesh_y + MW - 1) / MW, (mesh_x + rows - 1) / rows);
  if constexpr (lds)
    hipLaunchKernelGGL((k_conc_lds<P, C, R, NI>), g, blk, 0, stream, prm, phi, mu, (const R*)dphi, mulo, phi_o, mu_o,
                       mulo_o, tb, tsh);
  else
    hipLaunchKernelGGL((k_conc_march<P, C, R, NI>), g, blk, 0, stream, prm, phi, mu, (const R*)dphi, mulo, phi_o,
                       mu_o, mulo_o, tb, tsh);
}

// Fill the ghost layers of a freshly loaded state: every interior cell copies
// itself to its ghost images (apply_boundary_conditions(0) after loading).
template <class R>
__global__ void k_ghosts(const DevParams<R>* __restrict__ prm, R* __restrict__ phi, R* __restrict__ mu, int P, int C) {
  const DevParams<R>& p = *prm;
  const int y = 3 + blockIdx.x * BX + threadIdx.x;
  const int x = 3 + blockIdx.y * BY + threadIdx.y;
  if (x > p.mesh_x + 2 || y > p.mesh_y + 2) return;
  for (int a = 0; a < P; a++) {
    R* b = phi + (size_t)a * p.plane;
    write_with_ghosts(p, 0, b, x, y, b[(size_t)x * p.pitch + y]);
  }
  for (int k = 0; k < C; k++) {
    R* b = mu + (size_t)k * p.plane;
    write_with_ghosts(p, 1, b, x, y, b[(size_t)x * p.pitch + y]);
  }
}

// Moving frame (apply_shiftY, functions/shift.h:4-38): every padded column,
// ghost layers included, moves d rows towards y = 0 and the top d rows take
// the fill value of their plane.  Out of place, nf planes from src to dst.
struct ShiftFill {
  double v[GP_MAX_PHASES > GP_MAX_COMP ? GP_MAX_PHASES : GP_MAX_COMP];
};
template <class R>
__global__ void k_shift_y(const DevParams<R>* __restrict__ prm, const R* __restrict__ src, R* __restrict__ dst, int nf,
                          int d, ShiftFill f) {
  const DevParams<R>& p = *prm;
  const int y = blockIdx.x * BX + threadIdx.x;
  const int x = blockIdx.y * BY + threadIdx.y;
  if (x >= p.rx || y >= p.ry) return;
  for (int k = 0; k < nf; k++) {
    const size_t o = (size_t)k * p.plane + (size_t)x * p.pitch + y;
    dst[o] = y + d < p.ry ? src[o + d] : (R)f.v[k];
  }
}

// Interface position of the moving frame (check_SHIFT, functions/shift.h:44-66)
// over the interior rows: per row x, the largest padded y in [1, ry-1] at which
// the last phase goes from below 1/2 at y-1 to above 1/2 at y, 0 if none.  One
// block of IFB threads per row; the row result goes to out[x - 3].
constexpr int IFB = 256;
template <class R>
__global__ void __launch_bounds__(IFB) k_iface_rows(const DevParams<R>* __restrict__ prm, const R* __restrict__ phil,
                                                    int* __restrict__ out) {
  __shared__ int red[IFB];
  const DevParams<R>& p = *prm;
  const int x = 3 + blockIdx.x;
  const R* row = phil + (size_t)x * p.pitch;
  int best = 0;
  for (int y = 1 + threadIdx.x; y < p.ry; y += IFB) {
    const R a = row[y - 1], b = row[y];
    if ((a - (R(1) - a) < R(0)) && (b - (R(1) - b) > R(0))) best = max(best, y);
  }
  red[threadIdx.x] = best;
  __syncthreads();
  for (int s = IFB / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// interior <-> padded copies (host layout [f][MX][MY] dense, R or double)
template <class R, class S>
__global__ void k_pack(const DevParams<R>* __restrict__ prm, const S* __restrict__ src, R* __restrict__ dst, int nf) {
  const DevParams<R>& p = *prm;
  const int y = blockIdx.x * BX + threadIdx.x;
  const int x = blockIdx.y * BY + threadIdx.y;
  if (x >= p.mesh_x || y >= p.mesh_y) return;
  for (int f = 0; f < nf; f++)
    dst[(size_t)f * p.plane + (size_t)(x + 3) * p.pitch + (y + 3)] = (R)src[((size_t)f * p.mesh_x + x) * p.mesh_y + y];
}

template <class R, class S>
__global__ void k_unpack(const DevParams<R>* __restrict__ prm, const R* __restrict__ src, S* __restrict__ dst, int nf) {
  const DevParams<R>& p = *prm;
  const int y = blockIdx.x * BX + threadIdx.x;
  const int x = blockIdx.y * BY + threadIdx.y;
  if (x >= p.mesh_x || y >= p.mesh_y) return;
  for (int f = 0; f < nf; f++)
    dst[((size_t)f * p.mesh_x + x) * p.mesh_y + y] = (S)src[(size_t)f * p.plane + (size_t)(x + 3) * p.pitch + (y + 3)];
}

// Diagnostics: per-block partials (binary64) of max/min/sum of phi, max/min of mu,
// solute sum_a h_a c_a(mu) with half weights on the first and last interior
// node of each axis, and the count of non-finite values.
// Partial layout per block: [phi_max P][phi_min P][phi_sum P][mu_max C][mu_min C][solute C][nonfinite 1]
// Free-energy functional at interior node (x, y) in binary64, whatever the
// fields' precision.  The reference never sums it; its phase sweep is the
// variational derivative of eps a(phi, grad phi) + w(phi)/eps + sum_a h_a psi_a
// (dA/dphi: function_A_00.h:4-24, function_A_01.h:4-71; dw/dphi:
// functionW_01.h:6-39, functionW_02.h:4-33; psi: function_F_01_dpsi,
// functionF_01.h:39-57).  a = sum_{a<b} Gamma_ab a_c(q)^2 |q|^2 with
// q = R_ab (phi_a grad phi_b - phi_b grad phi_a) on the centred gradients of the
// phase sweep; w = 16/pi^2 sum Gamma_ab |phi_a phi_b| (obstacle) or
// 9 sum Gamma_ab phi_a^2 phi_b^2 (well), plus sum Gamma_abc |phi_a phi_b phi_c|.
// e[0] += eps a, e[1] += w / eps, e[2] += sum_a h_a psi_a, e[3] += sum_k mu_k c_k,
// each times wt dx dy.  T: the node's temperature (non-isothermal runs only).
template <int P, int C, class R>
__device__ __forceinline__ void node_energy(const DevParams<R>& p, const R* __restrict__ phi, const double* ph,
                                            const double* m, int x, int y, double T, double wt, double* e) {
  const double dx = (double)p.dx, dy = (double)p.dy;
  double cX[P], cY[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    const double f = (double)phi[idx(p, a, x + 1, y)], b = (double)phi[idx(p, a, x - 1, y)];
    const double r = (double)phi[idx(p, a, x, y + 1)], l = (double)phi[idx(p, a, x, y - 1)];
    cX[a] = 0.5 * ((f - ph[a]) / dx + (ph[a] - b) / dx);
    cY[a] = (r - l) / (2.0 * dy);
  }
  double ag = 0.0, wp = 0.0, w3 = 0.0;
#pragma unroll
  for (int a = 0; a < P; a++)
#pragma unroll
    for (int b = a + 1; b < P; b++) {
      double q[2] = {ph[a] * cX[b] - ph[b] * cX[a], ph[a] * cY[b] - ph[b] * cY[a]};
      double ac = 1.0;
      if (p.anisotropy) {
        const double u0 = q[0], u1 = q[1];
        q[0] = (double)p.rot[a][b][0][0] * u0 + (double)p.rot[a][b][0][1] * u1;
        q[1] = (double)p.rot[a][b][1][0] * u0 + (double)p.rot[a][b][1][1] * u1;
        const double qx2 = q[0] * q[0], qy2 = q[1] * q[1], q2 = qx2 + qy2;
        if (fabs(q2) > 1.0e-15) ac = 1.0 - (double)p.dab[a][b] * (3.0 - 4.0 * (qx2 * qx2 + qy2 * qy2) / (q2 * q2));
      }
      const double g = (double)p.gamma[a][b];
      ag += g * ac * ac * (q[0] * q[0] + q[1] * q[1]);
      wp += p.obstacle ? g * fabs(ph[a] * ph[b]) : g * ph[a] * ph[a] * ph[b] * ph[b];
#pragma unroll
      for (int c = b + 1; c < P; c++) w3 += (double)p.gamma_abc[a][b][c] * fabs(ph[a] * ph[b] * ph[c]);
    }
  const double wpot = (p.obstacle ? 16.0 / (M_PI * M_PI) : 9.0) * wp + w3;
  double bulk = 0.0, muc = 0.0;
#pragma unroll
  for (int a = 0; a < P; a++) {
    double s1 = 0.0;
#pragma unroll
    for (int b = 0; b < P; b++)
#pragma unroll
      for (int c = 0; c < P; c++)
        if (b != a && c != a && b < c) s1 += ph[b] * ph[c];
    const double h = 3.0 * ph[a] * ph[a] - 2.0 * ph[a] * ph[a] * ph[a] + 2.0 * ph[a] * s1;
    double c[C], psi = 0.0;
#pragma unroll
    for (int k = 0; k < C; k++) {
      double ck = 0.0;
#pragma unroll
      for (int l = 0; l < C; l++) {
        // Beq + dBbdT (T - Teq): at the node's temperature, or the run's table
        const double bs = p.ni ? (double)p.Beq[a][l] + (double)p.dBbdT[a][l] * (T - (double)p.Teq) : (double)p.Bsh[a][l];
        ck += (double)p.cmu[a][k][l] * (m[l] - bs);
      }
      c[k] = ck;
      psi -= m[k] * ck;
      muc += h * m[k] * ck;
    }
    // f_a(c) with B and C at T (isothermal: the run's tables)
    double fa = 0.0;
#pragma unroll
    for (int i = 0; i < C; i++) {
#pragma unroll
      for (int j = 0; j < C; j++)
        if (i <= j) fa += (double)p.A[a][i][j] * c[i] * c[j];
      fa += (p.ni ? (double)B_of_T<C>(p, P - 1, (R)T, i, a) : (double)p.B[a][i]) * c[i];
    }
    fa += p.ni ? (double)C_of_T<C>(p, P - 1, (R)T, a) : (double)p.Cf[a];
    psi += fa;
    bulk += h * psi;
  }
  const double v = wt * dx * dy;
  e[0] += v * ((double)p.epsilon * ag);
  e[1] += v * (wpot / (double)p.epsilon);
  e[2] += v * bulk;
  e[3] += v * muc;
}

template <int P, int C, class R>
__global__ void __launch_bounds__(256) k_stats(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                               const R* __restrict__ mu, const R* __restrict__ phi_prev,
                                               const R* __restrict__ mu_prev, double* __restrict__ part,
                                               double tb) {
  const DevParams<R>& p = *prm;
  constexpr int NE = 3 * P + 3 * C + 1 + P + C;  // first energy accumulator
  constexpr int NV = NE + 4;
  double acc[NV];
#pragma unroll
  for (int a = 0; a < P; a++) { acc[a] = -INFINITY; acc[P + a] = INFINITY; acc[2 * P + a] = 0.0; }
#pragma unroll
  for (int k = 0; k < C; k++) { acc[3 * P + k] = -INFINITY; acc[3 * P + C + k] = INFINITY; acc[3 * P + 2 * C + k] = 0.0; }
  acc[3 * P + 3 * C] = 0.0;
#pragma unroll
  for (int v = 3 * P + 3 * C + 1; v < NV; v++) acc[v] = 0.0;
  const long ncell = (long)p.mesh_x * p.mesh_y;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < ncell; i += (long)gridDim.x * blockDim.x) {
    int x = (int)(i / p.mesh_y) + 3, y = (int)(i % p.mesh_y) + 3;
    double w = ((x == 3 || x == p.mesh_x + 2) ? 0.5 : 1.0) * ((y == 3 || y == p.mesh_y + 2) ? 0.5 : 1.0);
    R ph[P], m[C];
#pragma unroll
    for (int a = 0; a < P; a++) {
      ph[a] = phi[idx(p, a, x, y)];
      double d = (double)ph[a];
      if (!isfinite(d)) acc[3 * P + 3 * C] += 1.0;
      if (phi_prev) {
        double e = d - (double)phi_prev[idx(p, a, x, y)];
        acc[3 * P + 3 * C + 1 + a] += e * e;
      }
      acc[a] = fmax(acc[a], d);
      acc[P + a] = fmin(acc[P + a], d);
      acc[2 * P + a] += d;
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      m[k] = mu[idx(p, k, x, y)];
      double d = (double)m[k];
      if (!isfinite(d)) acc[3 * P + 3 * C] += 1.0;
      if (mu_prev) {
        double e = d - (double)mu_prev[idx(p, k, x, y)];
        acc[3 * P + 3 * C + 1 + P + k] += e * e;
      }
      acc[3 * P + k] = fmax(acc[3 * P + k], d);
      acc[3 * P + C + k] = fmin(acc[3 * P + C + k], d);
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      double s = 0.0;
#pragma unroll
      for (int a = 0; a < P; a++) {
        double ca = 0.0;
#pragma unroll
        for (int l = 0; l < C; l++) {
          // non-isothermal: Beq + dBbdT (T - Teq) at the row's temperature
          const double bs = p.ni ? (double)p.Beq[a][l] + (double)p.dBbdT[a][l] * ((tb + (double)y * (double)p.tgG) - (double)p.Teq)
                                 : (double)p.Bsh[a][l];
          ca += (double)p.cmu[a][k][l] * ((double)m[l] - bs);
        }
        double pa = ph[a];
        double s1 = 0.0;
#pragma unroll
        for (int b = 0; b < P; b++)
#pragma unroll
          for (int c = 0; c < P; c++)
            if (b != a && c != a && b < c) s1 += (double)ph[b] * (double)ph[c];
        double h = 3.0 * pa * pa - 2.0 * pa * pa * pa + 2.0 * pa * s1;
        s += h * ca;
      }
      acc[3 * P + 2 * C + k] += w * s;
    }
    {
      double phd[P], md[C];
#pragma unroll
      for (int a = 0; a < P; a++) phd[a] = (double)ph[a];
#pragma unroll
      for (int k = 0; k < C; k++) md[k] = (double)m[k];
      const double T = p.ni ? tb + (double)y * (double)p.tgG : 0.0;  // unused when isothermal
      node_energy<P, C, R>(p, phi, phd, md, x, y, T, w, &acc[NE]);
    }
  }
  // block reduction through LDS
  __shared__ double red[256];
  for (int v = 0; v < NV; v++) {
    red[threadIdx.x] = acc[v];
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) {
        double o = red[threadIdx.x + s], me = red[threadIdx.x];
        bool ismax = (v < P) || (v >= 3 * P && v < 3 * P + C);
        bool ismin = (v >= P && v < 2 * P) || (v >= 3 * P + C && v < 3 * P + 2 * C);
        red[threadIdx.x] = ismax ? fmax(me, o) : ismin ? fmin(me, o) : me + o;
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)blockIdx.x * NV + v] = red[0];
    __syncthreads();
  }
}

// One pre-loop smoothing sweep over the interior (smooth(), solverloop.h:72-90):
// delta-phi of a cell enters only its own update, so each thread does both.
template <int P, int C, class R>
__global__ void __launch_bounds__(BX * BY) GP_HEAVY k_smooth(const DevParams<R>* __restrict__ prm, const R* __restrict__ phi,
                                                    const R* __restrict__ mu, const R* __restrict__ mulo,
                                                    R* __restrict__ phi_o, R* __restrict__ mu_o,
                                                    R* __restrict__ mulo_o) {
  const DevParams<R>& p = *prm;
  const int y = 3 + blockIdx.x * BX + threadIdx.x;
  const int x = 3 + blockIdx.y * BY + threadIdx.y;
  if (x > p.mesh_x + 2 || y > p.mesh_y + 2) return;
  R v[P][3][3];
  load3x3<P>(p, phi, x, y, v);
  Nbhd<P, R> n;
  make_nbhd<P>(p, v, n);
  R dp[P];
  cell_dphi_smooth<P, C>(p, n, dp);
  R phc[P], phf[P], phb[P], phr[P], phl[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    phc[a] = v[a][1][1];
    phf[a] = v[a][2][1];
    phb[a] = v[a][0][1];
    phr[a] = v[a][1][2];
    phl[a] = v[a][1][0];
  }
  R mc[C], mf[C], mb[C], mr[C], ml[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    mc[k] = mu[idx(p, k, x, y)];
    mf[k] = mu[idx(p, k, x + 1, y)];
    mb[k] = mu[idx(p, k, x - 1, y)];
    mr[k] = mu[idx(p, k, x, y + 1)];
    ml[k] = mu[idx(p, k, x, y - 1)];
  }
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
  R muo[C], dmu[C];
  cell_update_smooth<P, C>(p, phc, mc, Dmf, Dmb, Dmr, Dml, gmf, gmb, gmr, gml, muo, dmu);
#pragma unroll
  for (int a = 0; a < P; a++) write_with_ghosts(p, 0, phi_o + (size_t)a * p.plane, x, y, phc[a] + dp[a]);
  if constexpr (Ops<R>::Exact) {
#pragma unroll
    for (int k = 0; k < C; k++) write_with_ghosts(p, 1, mu_o + (size_t)k * p.plane, x, y, muo[k]);
  } else {
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

}  // namespace GPK_NS
