// gp_cell.hpp -- per-cell and per-face arithmetic of the grand-potential 2-D step
// for gfx950, templated on the phase count P, the independent-component count C
// and the real type R.
//
// Every function evaluates its value with the same sequence of IEEE operations
// as the reference serial solver (file:line cited per function), so the binary64
// instantiation compiled with -ffp-contract=off reproduces the reference bit for
// bit.  The binary32 instantiation runs the same sequence in float with the
// divisions by constant spacings replaced by multiplications (Exact = false).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "gpstep.h"

// The step kernels are compiled twice for binary64: in namespace gpk with the
// spacings' power-of-two test at run time, and, with -DGP_POW2 -DGPK_NS=gpk2,
// for spacings that are powers of two, where every division by dx, dy or 2 dy
// is an exact multiplication by the inverse (the run-time test and its
// branches cost 18% of the two-pass step at 1024^2 with four phases; the
// dispatcher takes this build for P <= 4).
#ifndef GPK_NS
#define GPK_NS gpk
#endif

namespace GPK_NS {

constexpr int PM = GP_MAX_PHASES;
constexpr int CM = GP_MAX_COMP;

// Constant tables the kernels read (device memory; indices are compile-time
// constants after unrolling, so the loads are scalar).
template <class R>
struct DevParams {
  long plane;             // elements per field plane (rows_x * pitch)
  int rx, ry, pitch;      // padded extents (MESH+6) and row pitch
  int mesh_x, mesh_y;
  int obstacle, anisotropy, mu_solver;
  int yskip;              // padded y index MESH_Y-2 whose y-face antitrapping is skipped
  int pair_sym;           // dab, rot and rot_inv are symmetric in the phase pair
  int pow2_dx, pow2_dy;   // spacing is a power of two (division = exact multiplication)
  int gsrc[2][2][6];      // [field][axis][ghost slot] -> padded source index (slots: 0,1,2,n-3,n-2,n-1)
  int gfree[2][2][2];     // [field][axis]: indices lo..hi of that axis are the source of no ghost of the field
  R dx, dy, dt, two_dy;
  R inv_dx, inv_dy, inv_two_dy;
  R epsilon, inv_eps, tau;
  R w_pref;               // 16/(pi*pi) (obstacle) or 9.0 (well)
  R jscale;               // (-0.25*M_PI*epsilon) or (-1.0*epsilon)
  R well_at;              // 0.5/sqrt(2.0)
  R diff_s, diff_l;       // DIFFUSIVITY of phase 0 and of the liquid, component 0 (adjoint)
  R gamma[PM][PM];
  R gamma_abc[PM][PM][PM];
  R tau_ab[PM][PM];
  R dab[PM][PM];
  R rot[PM][PM][2][2];
  R rot_inv[PM][PM][2][2];
  R at_coef[PM][CM];      // 1.0 - D_a[k][k]/D_liq[k][k]
  R dcm[PM][CM][CM][CM];  // Diffusivity[b][i][k]*cmu[b][k][j] at [b][i][j][k]
  R Dm_bulk[PM][CM][CM];  // face mobility between two cells one-hot in phase a (cell_D of the one-hot vector, face mean)
  R A[PM][CM][CM];
  R cmu[PM][CM][CM];
  R Bsh[PM][CM];          // Beq + dBbdT*(T-Teq)
  R B[PM][CM];
  R Cf[PM];
  // non-isothermal runs: the temperature of padded row Y is tb + Y*tgG, tb per step
  int ni;
  int tsrc[6];            // y ghost rows 0,1,2, ry-3, ry-2, ry-1 -> row their temperature copy reads (-1: none)
  R tgG, tgv;             // DeltaT*dy/Distance, velocity (Tempgrady)
  R Teq;
  R Beq[PM][CM], dBbdT[PM][CM];
  R dTs[PM], dTl[PM], dC[PM][CM];   // DELTA_T[a][a], DELTA_T[a][liquid], DELTA_C[a]
  R ceqL[PM][CM], ceqS[PM][CM];     // ceq[a][liquid], ceq[a][a]
  // MPI solver semantics (GP_MPI_* bits of gp_params.mpi; binary64 only)
  int mpi;
  R V;                    // molar volume: dpsi / V
  R noise4amp;            // 4.0 * Amp_Noise_Phase (the MPI noise amplitude)
  int mpi_noise;          // GP_MPI_NOISE and Noise_phasefield
  R* comp;                // composition planes [C][rows_x][pitch] (GP_MPI_COMPOSITION), else null
  unsigned long long* rstate;            // drand48 state before this step's draws
  unsigned long long lcg[34][2];         // drand48 map applied 2^k times: x -> lcg[k][0] x + lcg[k][1]
  unsigned long long lcg_step[2];        // the map of one step's (rows_x-2)(rows_y-2) draws
};

// The parameters of one phase, a, for cell_update of a cell that holds that phase
// alone: cell_update<1> and the functions it calls take DevParams or this view of
// it, in which every phase index stands for a.  The phase may differ from lane to
// lane, so the entries come through vector loads (a few KB, resident in L1) where
// DevParams' come through scalar ones.
template <class T>
struct PhaseRow {
  const T* t;
  int a;
  __device__ __forceinline__ const T& operator[](int) const { return t[a]; }
};

template <class R>
struct PhaseParams {
  const int &mu_solver, &pow2_dx, &pow2_dy;
  const R &dx, &dy, &dt, &inv_dx, &inv_dy, &jscale, &Teq, &tgv;
  PhaseRow<R[CM]> Bsh, Beq, dBbdT;
  PhaseRow<R[CM][CM]> A, cmu;
  __device__ __forceinline__ PhaseParams(const DevParams<R>& f, int a)
      : mu_solver(f.mu_solver), pow2_dx(f.pow2_dx), pow2_dy(f.pow2_dy), dx(f.dx), dy(f.dy), dt(f.dt),
        inv_dx(f.inv_dx), inv_dy(f.inv_dy), jscale(f.jscale), Teq(f.Teq), tgv(f.tgv), Bsh{f.Bsh, a}, Beq{f.Beq, a},
        dBbdT{f.dBbdT, a}, A{f.A, a}, cmu{f.cmu, a} {}
};

// drand48's generator: x' = (0x5DEECE66D x + 0xB) mod 2^48, value x' 2^-48
// (POSIX; glibc's erand48_r builds the double from the 48 bits, so the value is
// exact).
constexpr unsigned long long kLcgMask = (1ull << 48) - 1;

// The value of draw j >= 1 after state s: the map applied j times.
template <class R>
__device__ __forceinline__ double lcg_draw(const DevParams<R>& p, unsigned long long s, unsigned long long j) {
  unsigned long long A = 1, Cc = 0;
  for (int k = 0; k < 34 && (j >> k); k++)
    if ((j >> k) & 1ull) {
      Cc = (p.lcg[k][0] * Cc + p.lcg[k][1]) & kLcgMask;
      A = (p.lcg[k][0] * A) & kLcgMask;
    }
  return (double)((A * s + Cc) & kLcgMask) * 0x1p-48;
}

template <class R>
struct Ops;
template <>
struct Ops<double> {
  static constexpr bool Exact = true;
};
template <>
struct Ops<float> {
  static constexpr bool Exact = false;
};

// Division by a grid spacing.  When the spacing is a power of two, v/d and
// v*(1/d) round the same real number, so the multiplication is exact; the
// binary64 path divides otherwise.
template <class R, class Pm>
__device__ __forceinline__ R div_dx(R v, const Pm& p) {
  #ifdef GP_POW2
  return v * p.inv_dx;
#else
  if constexpr (Ops<R>::Exact) return p.pow2_dx ? v * p.inv_dx : v / p.dx; else return v * p.inv_dx;
#endif
}
template <class R, class Pm>
__device__ __forceinline__ R div_dy(R v, const Pm& p) {
  #ifdef GP_POW2
  return v * p.inv_dy;
#else
  if constexpr (Ops<R>::Exact) return p.pow2_dy ? v * p.inv_dy : v / p.dy; else return v * p.inv_dy;
#endif
}
template <class R>
__device__ __forceinline__ R div_2dy(R v, const DevParams<R>& p) {
  #ifdef GP_POW2
  return v * p.inv_two_dy;
#else
  if constexpr (Ops<R>::Exact) return p.pow2_dy ? v * p.inv_two_dy : v / p.two_dy; else return v * p.inv_two_dy;
#endif
}

// sqrt that skips the evaluation for an exact zero argument (sqrt(+0) = +0)
template <class R>
__device__ __forceinline__ R sqrt_nz(R v) {
  return v == R(0) ? R(0) : sqrt(v);
}

// ---------------------------------------------------------------- thermodynamics

// c_a,i(mu)  (functionF_01.h:30-37)
template <int C, class R, class Pm>
__device__ __forceinline__ R c_mu(const Pm& p, const R* mu, int a, int i) {
  R s = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) s += p.cmu[a][i][k] * (mu[k] - p.Bsh[a][k]);
  return s;
}

// Mu_a,i(c)  (functionF_01.h:19-29)
template <int C, class R, class Pm>
__device__ __forceinline__ R Mu_of_c(const Pm& p, const R* c, int a, int i) {
  R s = R(2.0) * p.A[a][i][i] * c[i] + p.Bsh[a][i];
#pragma unroll
  for (int j = 0; j < C; j++)
    if (i != j) s += p.A[a][i][j] * c[j];
  return s;
}

// f_a(c)  (functionF_01.h:5-18)
template <int C, class R>
__device__ __forceinline__ R free_energy(const DevParams<R>& p, const R* c, int a) {
  R s = R(0);
#pragma unroll
  for (int i = 0; i < C; i++) {
#pragma unroll
    for (int j = 0; j < C; j++)
      if (i <= j) s += p.A[a][i][j] * c[i] * c[j];
    s += p.B[a][i] * c[i];
  }
  s += p.Cf[a];
  return s;
}

// h_a(phi)  (functionH.h:24-36)
template <int P, class R>
__device__ __forceinline__ R hphi(const R* ph, int a) {
  R s1 = R(0);
  R s = R(3.0) * ph[a] * ph[a] - R(2.0) * ph[a] * ph[a] * ph[a];
#pragma unroll
  for (int b = 0; b < P; b++)
#pragma unroll
    for (int c = 0; c < P; c++)
      if (b != a && c != a && b < c) s1 += ph[b] * ph[c];
  s1 *= R(2.0) * ph[a];
  return s + s1;
}

// d h_b / d phi_a  (functionH.h:1-23)
template <int P, class R>
__device__ __forceinline__ R dhphi(const R* ph, int b, int a) {
  R s = R(0);
  if (a == b) {
    s = R(6.0) * ph[a] * (R(1.0) - ph[a]);
#pragma unroll
    for (int e = 0; e < P; e++)
#pragma unroll
      for (int f = 0; f < P; f++)
        if (e != b && f != b && e < f) s += R(2.0) * ph[e] * ph[f];
  } else {
#pragma unroll
    for (int e = 0; e < P; e++)
      if (e != b && e != a) s += R(2.0) * ph[e];
    s *= ph[b];
  }
  return s;
}

// psi_b(mu) = f_b(c_b(mu)) - mu.c_b(mu)  (functionF_01.h:41-57, the b-term of dpsi)
template <int C, class R>
__device__ __forceinline__ R psi_of_mu(const DevParams<R>& p, const R* mu, int b) {
  R c[C];
  R psi = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    c[k] = c_mu<C>(p, mu, b, k);
    psi -= mu[k] * c[k];
  }
  psi += free_energy<C>(p, c, b);
  return psi;
}

// tau(phi)  (functionTau.h:1-16)
template <int P, class R>
__device__ __forceinline__ R tau_phi(const DevParams<R>& p, const R* ph) {
  R s = R(0), s1 = R(0);
#pragma unroll
  for (int a = 0; a < P; a++)
#pragma unroll
    for (int b = 0; b < P; b++)
      if (a < b) {
        s += p.tau_ab[a][b] * ph[a] * ph[b];
        s1 += ph[a] * ph[b];
      }
  if (s1 != R(0)) return s / s1;
  return p.tau;
}

// ---------------------------------------------------------------- temperature

// Non-isothermal runs (ISOTHERMAL = 0): temperature of padded row y,
// temp_bottom + Y*GRADIENT (functions/Temperature_gradient.h:17-19), where Y is
// the row itself or, when proxy is set and the row is a ghost row with a
// temperature boundary copy, the row it copies (boundary_serial.h:176-203).
// In the step after a moving-frame shift by tsh rows the temperature was moved
// with the fields (functions/shift.h:19): row Y then holds the value of row
// Y + tsh of the profile before the shift, except the top tsh rows, which keep
// their own.
template <class R>
__device__ __forceinline__ R temp_row(const DevParams<R>& p, R tb, int y, bool proxy, int tsh = 0) {
  int Y = y;
  if (proxy) {
    if (y <= 2 && p.tsrc[y] >= 0) Y = p.tsrc[y];
    else if (y >= p.ry - 3 && p.tsrc[3 + y - (p.ry - 3)] >= 0) Y = p.tsrc[3 + y - (p.ry - 3)];
  }
  if (Y < p.ry - tsh) Y += tsh;
  return tb + (R)Y * p.tgG;
}

// Beq + dBbdT (T - Teq) of c_a(mu) and Mu_a(c) at temperature T (functionF_01.h:19-37)
template <class R, class Pm>
__device__ __forceinline__ R bsh_t(const Pm& p, int a, int k, R T) {
  return p.Beq[a][k] + p.dBbdT[a][k] * (T - p.Teq);
}

template <int C, class R, class Pm>
__device__ __forceinline__ R c_mu_t(const Pm& p, const R* mu, int a, int i, R T) {
  R s = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) s += p.cmu[a][i][k] * (mu[k] - bsh_t(p, a, k, T));
  return s;
}

template <int C, class R, class Pm>
__device__ __forceinline__ R Mu_of_c_t(const Pm& p, const R* c, int a, int i, R T) {
  R s = R(2.0) * p.A[a][i][i] * c[i] + bsh_t(p, a, i, T);
#pragma unroll
  for (int j = 0; j < C; j++)
    if (i != j) s += p.A[a][i][j] * c[j];
  return s;
}

// B_a,i(T) and C_a(T) (functionF_01.h:62-104), the tables init_propertymatrices(T)
// leaves for the phase-field terms of a cell of temperature T
template <int C, class R>
__device__ __forceinline__ R B_of_T(const DevParams<R>& p, int L, R T, int i, int a) {
  if (a == L) return R(0);
  R cl[C], cs[C], sum_c = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    cl[k] = p.ceqL[a][k] - (p.dC[a][k]) * (p.Teq - T) / (p.dTl[a]);
    cs[k] = p.ceqS[a][k] - (p.dC[a][k]) * (p.Teq - T) / (p.dTs[a]);
    if (k != i) sum_c += p.A[L][k][i] * cl[k] - p.A[a][k][i] * cs[k];
  }
  return (R(2.0) * (p.A[L][i][i] * cl[i] - p.A[a][i][i] * cs[i]) + sum_c);
}

template <int C, class R>
__device__ __forceinline__ R C_of_T(const DevParams<R>& p, int L, R T, int a) {
  if (a == L) return R(0);
  R cl[C], cs[C], sum_c = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    cl[k] = p.ceqL[a][k] - (p.dC[a][k]) * (p.Teq - T) / (p.dTl[a]);
    cs[k] = p.ceqS[a][k] - (p.dC[a][k]) * (p.Teq - T) / (p.dTs[a]);
  }
#pragma unroll
  for (int i = 0; i < C; i++)
#pragma unroll
    for (int j = 0; j < C; j++)
      if (i <= j) sum_c += (p.A[a][i][j] * cs[i] * cs[j] - p.A[L][i][j] * cl[i] * cl[j]);
  return sum_c;
}

template <int P, int C, class R>
__device__ __forceinline__ R psi_of_mu_t(const DevParams<R>& p, const R* mu, int b, R T) {
  R c[C];
  R psi = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    c[k] = c_mu_t<C>(p, mu, b, k, T);
    psi -= mu[k] * c[k];
  }
  // free energy with B(T), C(T)
  R f = R(0);
#pragma unroll
  for (int i = 0; i < C; i++) {
#pragma unroll
    for (int j = 0; j < C; j++)
      if (i <= j) f += p.A[b][i][j] * c[i] * c[j];
    f += B_of_T<C>(p, P - 1, T, i, b) * c[i];
  }
  f += C_of_T<C>(p, P - 1, T, b);
  psi += f;
  return psi;
}

// the same functions at the run's temperature (tables) or, with NI, at T
template <int C, bool NI, class R, class Pm>
__device__ __forceinline__ R c_mu_(const Pm& p, const R* mu, int a, int i, R T) {
  if constexpr (NI) return c_mu_t<C>(p, mu, a, i, T);
  else return c_mu<C>(p, mu, a, i);
}
template <int C, bool NI, class R, class Pm>
__device__ __forceinline__ R Mu_of_c_(const Pm& p, const R* c, int a, int i, R T) {
  if constexpr (NI) return Mu_of_c_t<C>(p, c, a, i, T);
  else return Mu_of_c<C>(p, c, a, i);
}
template <int P, int C, bool NI, class R>
__device__ __forceinline__ R psi_of_mu_(const DevParams<R>& p, const R* mu, int b, R T) {
  if constexpr (NI) return psi_of_mu_t<P, C>(p, mu, b, T);
  else return psi_of_mu<C>(p, mu, b);
}

// ---------------------------------------------------------------- anisotropy

// 2-D block of multiply(R, q) (matrix.h:22-33, DIMENSION = 2)
template <class R>
__device__ __forceinline__ void rot2(const R (&M)[2][2], const R* q, R* out) {
#pragma unroll
  for (int i = 0; i < 2; i++) {
    R s = R(0);
    s = s + M[i][0] * q[0];
    s = s + M[i][1] * q[1];
    out[i] = s;
  }
}

// a_c(q) of the four-fold cubic form  (anisotropy_01.h:29-48)
template <class R>
__device__ __forceinline__ R ac_of_q(R dab, const R* q) {
  R qx2 = q[0] * q[0], qx4 = qx2 * qx2, qy2 = q[1] * q[1], qy4 = qy2 * qy2;
  R q2 = qx2 + qy2;
  if (fabs(q2) > R(1.0e-15)) return R(1.0) - dab * (R(3.0) - R(4.0) * (qx4 + qy4) / (q2 * q2));
  return R(1.0);
}

// d a_c / d q  (anisotropy_01.h:9-27)
template <class R>
__device__ __forceinline__ void dadq_of_q(R dab, const R* q, R* d) {
  R qx3 = q[0] * q[0] * q[0], qy3 = q[1] * q[1] * q[1];
  R q2 = q[0] * q[0] + q[1] * q[1];
  R q22 = q2 * q2, q23 = q2 * q2 * q2;
  R q4 = qx3 * q[0] + qy3 * q[1];
  if (fabs(q2) > R(1.0e-15)) {
    if constexpr (Ops<R>::Exact) {
      d[0] = R(16.0) * dab * (qx3 / q22 - q[0] * q4 / q23);
      d[1] = R(16.0) * dab * (qy3 / q22 - q[1] * q4 / q23);
    } else {
      // binary32: |q|^6 is subnormal for |q|^2 < 2.3e-13 and rounds to zero
      // just above the 1e-15 guard, which made q4 / q23 infinite; the same
      // quantity is q * (q4 / |q|^4) / |q|^2 with q4 / |q|^4 in [1/2, 1]
      (void)q23;
      const R r = q4 / q22;
      d[0] = R(16.0) * dab * (qx3 / q22 - q[0] * r / q2);
      d[1] = R(16.0) * dab * (qy3 / q22 - q[1] * r / q2);
    }
  } else {
    d[0] = R(0);
    d[1] = R(0);
  }
}

// ---------------------------------------------------------------- neighbourhood

// phi gradients around one cell, from the 3x3 block v[a][i][j] (i,j = 0..2 for
// offsets -1..+1); the formulas are calculate_gradients.h:108-128.
template <int P, class R>
struct Nbhd {
  R ph[P];                 // phi at the cell
  R gXc[P], gXb[P];        // x-face gradients at faces (x|x+1), (x-1|x)
  R sXc[P], sXb[P];        // x-face averages
  R gYc[P], gYl[P];        // y-face gradients at faces (y|y+1), (y-1|y)
  R sYc[P], sYl[P];
  R cXc[P], cYc[P];        // centred gradients at the cell
  R cYf[P], cYb[P];        // centred y-gradients at (x+1,y), (x-1,y)
  R cXr[P], cXl[P];        // centred x-gradients at (x,y+1), (x,y-1)
  bool present[P];         // phase b is nonzero somewhere in the 3x3 block
};

template <int P, class R>
__device__ __forceinline__ void make_nbhd(const DevParams<R>& p, const R (&v)[P][3][3], Nbhd<P, R>& n) {
#pragma unroll
  for (int a = 0; a < P; a++) {
    bool nz = false;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) nz = nz || (v[a][i][j] != R(0));
    n.present[a] = nz;
    n.ph[a] = v[a][1][1];
    n.gXc[a] = div_dx(v[a][2][1] - v[a][1][1], p);
    n.gXb[a] = div_dx(v[a][1][1] - v[a][0][1], p);
    n.sXc[a] = R(0.5) * (v[a][2][1] + v[a][1][1]);
    n.sXb[a] = R(0.5) * (v[a][1][1] + v[a][0][1]);
    n.gYc[a] = div_dy(v[a][1][2] - v[a][1][1], p);
    n.gYl[a] = div_dy(v[a][1][1] - v[a][1][0], p);
    n.sYc[a] = R(0.5) * (v[a][1][2] + v[a][1][1]);
    n.sYl[a] = R(0.5) * (v[a][1][1] + v[a][1][0]);
    n.cXc[a] = R(0.5) * (n.gXc[a] + n.gXb[a]);
    n.cYc[a] = div_2dy(v[a][1][2] - v[a][1][0], p);
    n.cYf[a] = div_2dy(v[a][2][2] - v[a][2][0], p);
    n.cYb[a] = div_2dy(v[a][0][2] - v[a][0][0], p);
    R gx_r = div_dx(v[a][2][2] - v[a][1][2], p), gx_rb = div_dx(v[a][1][2] - v[a][0][2], p);
    R gx_l = div_dx(v[a][2][0] - v[a][1][0], p), gx_lb = div_dx(v[a][1][0] - v[a][0][0], p);
    n.cXr[a] = R(0.5) * (gx_r + gx_rb);
    n.cXl[a] = R(0.5) * (gx_l + gx_lb);
  }
}

// ---------------------------------------------------------------- delta-phi

// dA/dphi_a  (function_A_00.h:4-24 isotropic; function_A_01.h:4-71 anisotropic)
template <int P, class R>
__device__ __forceinline__ R dAdphi(const DevParams<R>& p, const Nbhd<P, R>& n, int a) {
  if (!p.anisotropy) {
    R sum = R(0);
#pragma unroll
    for (int b = 0; b < P; b++) {
      if (b == a || !n.present[b]) continue;  // an absent phase contributes exact zeros
      R sp = R(0);
      sp += (n.ph[a] * n.cXc[b] - n.ph[b] * n.cXc[a]) * n.cXc[b];
      sp += (n.ph[a] * n.cYc[b] - n.ph[b] * n.cYc[a]) * n.cYc[b];
      sp *= p.gamma[a][b];
      sum += sp;
    }
    return R(2.0) * sum;
  }
  R sum1 = R(0), sum2 = R(0);
#pragma unroll
  for (int b = 0; b < P; b++) {
    if (b == a || !n.present[b]) continue;  // an absent phase contributes exact zeros
    R u[2], q[2], d[2], dq[2], rdq[2];
    u[0] = (n.ph[a] * n.cXc[b] - n.ph[b] * n.cXc[a]);
    u[1] = (n.ph[a] * n.cYc[b] - n.ph[b] * n.cYc[a]);
    rot2(p.rot[a][b], u, q);
    dadq_of_q(p.dab[a][b], q, d);
    R qab2 = (q[0] * q[0] + q[1] * q[1]);
    R ac1 = ac_of_q(p.dab[a][b], q), ac2 = ac1 * ac1;
    dq[0] = n.cXc[b];
    dq[1] = n.cYc[b];
    rot2(p.rot[a][b], dq, rdq);
    R s1 = R(0), s2 = R(0);
    s1 += q[0] * rdq[0];
    s1 += q[1] * rdq[1];
    s2 += d[0] * rdq[0];
    s2 += d[1] * rdq[1];
    s1 *= p.gamma[a][b] * ac2;
    s2 *= p.gamma[a][b] * ac1 * qab2;
    sum1 += s1;
    sum2 += s2;
  }
  return R(2.0) * (sum1 + sum2);
}

// per-face data of the anisotropic divergence for pair (a,b)
template <class R>
struct FaceQ {
  R flux;      // sa*gb - sb*ga (unrotated normal component)
  R ac, ac2;   // a_c(q), a_c^2
  R q2;        // |q|^2
  R rd[2];     // R^-1 * da_c/dq
};

template <class R>
__device__ __forceinline__ void face_q(const DevParams<R>& p, int a, int b, R u0, R u1, R flux, FaceQ<R>& f) {
  R u[2] = {u0, u1}, q[2], d[2];
  rot2(p.rot[a][b], u, q);
  f.flux = flux;
  f.ac = ac_of_q(p.dab[a][b], q);
  f.ac2 = f.ac * f.ac;
  dadq_of_q(p.dab[a][b], q, d);
  rot2(p.rot_inv[a][b], d, f.rd);
  f.q2 = q[0] * q[0] + q[1] * q[1];
}

// div (dA / d grad phi_a)  (function_A_00.h:25-58 isotropic; function_A_01.h:101-219 anisotropic)
template <int P, class R>
__device__ __forceinline__ R divdAdgradphi(const DevParams<R>& p, const Nbhd<P, R>& n, int a) {
  if (!p.anisotropy) {
    R sum = R(0);
#pragma unroll
    for (int b = 0; b < P; b++) {
      if (b == a || !n.present[b]) continue;  // an absent phase contributes exact zeros
      R fc = n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a];
      R fb = n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a];
      R dv = div_dx(fc * (-n.sXc[b]) - (fb * (-n.sXb[b])), p);
      R gc = n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a];
      R gl = n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a];
      dv += div_dy(gc * (-n.sYc[b]) - (gl * (-n.sYl[b])), p);
      dv *= p.gamma[a][b];
      sum += dv;
    }
    return R(2.0) * sum;
  }
  R sum1 = R(0), sum2 = R(0);
#pragma unroll
  for (int b = 0; b < P; b++) {
    if (b == a || !n.present[b]) continue;  // an absent phase contributes exact zeros
    FaceQ<R> F, Bk, Rt, L;
    face_q(p, a, b, n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a],
           R(0.5) * (n.sXc[a] * (n.cYc[b] + n.cYf[b]) - n.sXc[b] * (n.cYc[a] + n.cYf[a])),
           n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a], F);
    face_q(p, a, b, n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a],
           R(0.5) * (n.sXb[a] * (n.cYb[b] + n.cYc[b]) - n.sXb[b] * (n.cYb[a] + n.cYc[a])),
           n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a], Bk);
    face_q(p, a, b, R(0.5) * (n.sYc[a] * (n.cXc[b] + n.cXr[b]) - n.sYc[b] * (n.cXc[a] + n.cXr[a])),
           n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a],
           n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a], Rt);
    face_q(p, a, b, R(0.5) * (n.sYl[a] * (n.cXl[b] + n.cXc[b]) - n.sYl[b] * (n.cXl[a] + n.cXc[a])),
           n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a],
           n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a], L);
    R d1 = div_dx((F.ac2 * F.flux * (-n.sXc[b])) - (Bk.ac2 * Bk.flux * (-n.sXb[b])), p);
    d1 += div_dy((Rt.ac2 * Rt.flux * (-n.sYc[b])) - (L.ac2 * L.flux * (-n.sYl[b])), p);
    d1 *= p.gamma[a][b];
    sum1 += d1;
    R d2 = div_dx(F.ac * F.q2 * F.rd[0] * (-n.sXc[b]) - Bk.ac * Bk.q2 * Bk.rd[0] * (-n.sXb[b]), p);
    d2 += div_dy(Rt.ac * Rt.q2 * Rt.rd[1] * (-n.sYc[b]) - L.ac * L.q2 * L.rd[1] * (-n.sYl[b]), p);
    d2 *= p.gamma[a][b];
    sum2 += d2;
  }
  return (R(2.0) * (sum1 + sum2) + R(0));
}

// dA/dphi_a and div(dA/dgrad phi_a) of the anisotropic form for every phase a
// with want[a], pair by pair.  With dab, rot and rot_inv symmetric in the
// pair, the ordered pair (b,a) sees the vector u of (a,b) negated: q = R u,
// da_c/dq and R^-1 da_c/dq change sign, a_c and |q|^2 do not (a_c is even in q,
// da_c/dq odd, and IEEE negation commutes with the products and sums involved).
// So the a_c, da_c/dq and face terms of each unordered pair are evaluated once
// and used with a sign for both phases.  Visiting pairs (a,b), a < b, in
// ascending order hands every phase its partners in ascending order, the order
// of dAdphi / divdAdgradphi above, so each per-phase sum is formed from the
// same terms in the same order.  Terms may differ from the per-phase functions
// only in the sign of a zero, which leaves nonzero sums unchanged; the results
// are returned as dA = 2(s1+s2) (entering lam as -dA + dG, where either zero
// gives +0) and dG = 2(s1+s2) + 0 (zero normalised as in divdAdgradphi).
template <int P, class R>
__device__ __forceinline__ void aniso_pairs(const DevParams<R>& p, const Nbhd<P, R>& n, const bool* want, R* dA,
                                            R* dG) {
  R a1[P], a2[P], g1[P], g2[P];
#pragma unroll
  for (int a = 0; a < P; a++) a1[a] = a2[a] = g1[a] = g2[a] = R(0);
#pragma unroll
  for (int a = 0; a < P; a++)
#pragma unroll
    for (int b = a + 1; b < P; b++) {
      const bool ua = want[a] && n.present[b], ub = want[b] && n.present[a];
      if (!ua && !ub) continue;
      // dA/dphi: q of the cell-centred u (function_A_01.h:4-71)
      {
        R u[2], q[2], d[2];
        u[0] = (n.ph[a] * n.cXc[b] - n.ph[b] * n.cXc[a]);
        u[1] = (n.ph[a] * n.cYc[b] - n.ph[b] * n.cYc[a]);
        rot2(p.rot[a][b], u, q);
        dadq_of_q(p.dab[a][b], q, d);
        R qab2 = (q[0] * q[0] + q[1] * q[1]);
        R ac1 = ac_of_q(p.dab[a][b], q), ac2 = ac1 * ac1;
        if (ua) {
          R dq[2] = {n.cXc[b], n.cYc[b]}, rdq[2];
          rot2(p.rot[a][b], dq, rdq);
          R s1 = R(0), s2 = R(0);
          s1 += q[0] * rdq[0];
          s1 += q[1] * rdq[1];
          s2 += d[0] * rdq[0];
          s2 += d[1] * rdq[1];
          s1 *= p.gamma[a][b] * ac2;
          s2 *= p.gamma[a][b] * ac1 * qab2;
          a1[a] += s1;
          a2[a] += s2;
        }
        if (ub) {
          R dq[2] = {n.cXc[a], n.cYc[a]}, rdq[2];
          rot2(p.rot[b][a], dq, rdq);
          R s1 = R(0), s2 = R(0);
          s1 += (-q[0]) * rdq[0];
          s1 += (-q[1]) * rdq[1];
          s2 += (-d[0]) * rdq[0];
          s2 += (-d[1]) * rdq[1];
          s1 *= p.gamma[b][a] * ac2;
          s2 *= p.gamma[b][a] * ac1 * qab2;
          a1[b] += s1;
          a2[b] += s2;
        }
      }
      // div(dA/dgrad phi): the four faces (function_A_01.h:101-219)
      FaceQ<R> F, Bk, Rt, L;
      face_q(p, a, b, n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a],
             R(0.5) * (n.sXc[a] * (n.cYc[b] + n.cYf[b]) - n.sXc[b] * (n.cYc[a] + n.cYf[a])),
             n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a], F);
      face_q(p, a, b, n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a],
             R(0.5) * (n.sXb[a] * (n.cYb[b] + n.cYc[b]) - n.sXb[b] * (n.cYb[a] + n.cYc[a])),
             n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a], Bk);
      face_q(p, a, b, R(0.5) * (n.sYc[a] * (n.cXc[b] + n.cXr[b]) - n.sYc[b] * (n.cXc[a] + n.cXr[a])),
             n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a],
             n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a], Rt);
      face_q(p, a, b, R(0.5) * (n.sYl[a] * (n.cXl[b] + n.cXc[b]) - n.sYl[b] * (n.cXl[a] + n.cXc[a])),
             n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a],
             n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a], L);
      if (ua) {
        R d1 = div_dx((F.ac2 * F.flux * (-n.sXc[b])) - (Bk.ac2 * Bk.flux * (-n.sXb[b])), p);
        d1 += div_dy((Rt.ac2 * Rt.flux * (-n.sYc[b])) - (L.ac2 * L.flux * (-n.sYl[b])), p);
        d1 *= p.gamma[a][b];
        g1[a] += d1;
        R d2 = div_dx(F.ac * F.q2 * F.rd[0] * (-n.sXc[b]) - Bk.ac * Bk.q2 * Bk.rd[0] * (-n.sXb[b]), p);
        d2 += div_dy(Rt.ac * Rt.q2 * Rt.rd[1] * (-n.sYc[b]) - L.ac * L.q2 * L.rd[1] * (-n.sYl[b]), p);
        d2 *= p.gamma[a][b];
        g2[a] += d2;
      }
      if (ub) {
        R d1 = div_dx((F.ac2 * (-F.flux) * (-n.sXc[a])) - (Bk.ac2 * (-Bk.flux) * (-n.sXb[a])), p);
        d1 += div_dy((Rt.ac2 * (-Rt.flux) * (-n.sYc[a])) - (L.ac2 * (-L.flux) * (-n.sYl[a])), p);
        d1 *= p.gamma[b][a];
        g1[b] += d1;
        R d2 = div_dx(F.ac * F.q2 * (-F.rd[0]) * (-n.sXc[a]) - Bk.ac * Bk.q2 * (-Bk.rd[0]) * (-n.sXb[a]), p);
        d2 += div_dy(Rt.ac * Rt.q2 * (-Rt.rd[1]) * (-n.sYc[a]) - L.ac * L.q2 * (-L.rd[1]) * (-n.sYl[a]), p);
        d2 *= p.gamma[b][a];
        g2[b] += d2;
      }
    }
#pragma unroll
  for (int a = 0; a < P; a++) {
    dA[a] = R(2.0) * (a1[a] + a2[a]);
    dG[a] = (R(2.0) * (g1[a] + g2[a]) + R(0));
  }
}

// dw/dphi_a  (functionW_01.h:6-39 obstacle, functionW_02.h:4-33 well)
template <int P, class R>
__device__ __forceinline__ R dwdphi(const DevParams<R>& p, const R* ph, const bool* act, int a) {
  R sum = R(0);
  if (p.obstacle) {
#pragma unroll
    for (int b = 0; b < P; b++)
      if (b != a && act[b]) {
        if ((ph[a] * ph[b]) >= R(0)) sum += p.gamma[a][b] * (ph[b]);
        else sum += -p.gamma[a][b] * (ph[b]);
      }
  } else {
#pragma unroll
    for (int b = 0; b < P; b++)
      if (b != a && act[b]) sum += R(2.0) * p.gamma[a][b] * (ph[b] * ph[b] * ph[a]);
  }
  sum *= p.w_pref;
#pragma unroll
  for (int b = 0; b < P; b++)
#pragma unroll
    for (int c = 0; c < P; c++)
      if (b != a && c != a && b < c && act[b] && act[c]) {
        R pbc = ph[b] * ph[c];
        if (ph[a] * pbc >= R(0)) sum += p.gamma_abc[a][b][c] * pbc;
        else sum += -p.gamma_abc[a][b][c] * pbc;
      }
  return sum;
}

// Gibbs-simplex projection  (simplex_projection.h:1-49)
template <int P, class R>
__device__ __forceinline__ void project_simplex(const R* ph, const bool* act, R* dp) {
  R Deltaphi = R(0), sum_phib = R(0);
  int count = 0;
#pragma unroll
  for (int a = 0; a < P; a++)
    if (act[a] && (ph[a] + dp[a]) > R(0) && (ph[a] + dp[a]) < R(1.0)) {
      count++;
      sum_phib += ph[a];
    }
#pragma unroll
  for (int a = 0; a < P; a++)
    if ((ph[a] + dp[a]) < R(0)) {
      R Da = fabs(dp[a] + ph[a]);
      // binary32: dp + |dp + ph| can leave ph + dp a few ulps above zero, and
      // the phase then takes a share Deltaphi * ph / sum_phib below, where a
      // tiny or negative sum_phib (phases at -1e-17 after earlier steps) made
      // that share 1e7 times Deltaphi and the fields non-finite a few steps
      // later; -ph is the exact value of dp + |dp + ph| here
      if constexpr (Ops<R>::Exact) dp[a] += Da;
      else dp[a] = -ph[a];
      Deltaphi += Da;
    }
  if (Deltaphi > R(0)) {
#pragma unroll
    for (int b = 0; b < P; b++)
      if (act[b] && ((ph[b] + dp[b]) > R(0)) && ((ph[b] + dp[b]) < R(1.0))) {
        if (fabs(sum_phib) > R(0)) dp[b] -= Deltaphi * (ph[b]) / (sum_phib);
        else dp[b] -= Deltaphi / R(count);
      }
  }
  bool done = false;
#pragma unroll
  for (int a = 0; a < P; a++)
    if (!done && act[a] && (ph[a] + dp[a]) > R(1.0)) {
      dp[a] = (R(1.0) - ph[a]);
#pragma unroll
      for (int b = 0; b < P; b++)
        if (act[b] && b != a) dp[b] = -ph[b];
      done = true;
    }
}

// Active phases of a cell: |div phi_a| > 0 (calculate_divergence_phasefield.h:9-16).
// Returns whether any phase is active.
template <int P, class R>
__device__ __forceinline__ bool cell_active(const DevParams<R>& p, const Nbhd<P, R>& n, bool* act) {
  bool any = false;
#pragma unroll
  for (int a = 0; a < P; a++) {
    R divphi = div_dx(n.gXc[a] - n.gXb[a], p);
    divphi += div_dy(n.gYc[a] - n.gYl[a], p);
    act[a] = fabs(divphi) > R(0);
    any = any || act[a];
  }
  return any;
}

// delta-phi of one cell from its active set; with `pairs`, dA / dG hold the
// anisotropic dA/dphi and div(dA/dgrad phi) of every active phase, else they
// are evaluated here phase by phase  (calculate_divergence_phasefield.h:4-62)
// nzw (phase-field noise): the glibc rand() words of the cell's active phases
// in phase order, amp = Amp_Noise_Phase; nullptr without noise.
// With MPI (the MPI solver's semantics, binary64): the driving force is
// dpsi / V under GP_MPI_DPSI_V, and mnz (4 Amp drand48() of the cell) adds
// mnz phi_a (1 - phi_a) dpsi / V under p.mpi_noise
// (MPI calculate_divergence_phasefield.h:335-343).
template <int P, int C, class R, bool NI = false, bool MPI = false>
__device__ __forceinline__ void cell_dphi_rest(const DevParams<R>& p, const Nbhd<P, R>& n, const R* mu,
                                               const bool* act, bool any, bool pairs, R* dA, R* dG, R* dp,
                                               R T = R(0), const uint32_t* nzw = nullptr, R amp = R(0),
                                               R mnz = R(0)) {
  R lam[P], psi[P];
#pragma unroll
  for (int a = 0; a < P; a++) dp[a] = R(0);
  if (any) {
#pragma unroll
    for (int b = 0; b < P; b++) psi[b] = psi_of_mu_<P, C, NI>(p, mu, b, T);
    R sl = R(0);
    int active = 0;
#pragma unroll
    for (int a = 0; a < P; a++)
      if (act[a]) {
        R dps = R(0);
#pragma unroll
        for (int b = 0; b < P; b++) dps += psi[b] * dhphi<P>(n.ph, b, a);
        if (!pairs) {
          dA[a] = dAdphi<P>(p, n, a);
          dG[a] = divdAdgradphi<P>(p, n, a);
        }
        if constexpr (MPI) {
          lam[a] = p.epsilon * (-dA[a] + dG[a]) - p.inv_eps * dwdphi<P>(p, n.ph, act, a) -
                   ((p.mpi & GP_MPI_DPSI_V) ? dps / p.V : dps);
          if (p.mpi_noise) lam[a] += mnz * n.ph[a] * (R(1.0) - n.ph[a]) * dps / p.V;
        } else {
          lam[a] = p.epsilon * (-dA[a] + dG[a]) - p.inv_eps * dwdphi<P>(p, n.ph, act, a) - dps;
        }
        // AMP * rand() / RAND_MAX * phi_a (1 - phi_a)  (calculate_divergence_phasefield.h:33-35)
        if (nzw) lam[a] += amp * ((R)(nzw[active] >> 1) / (R)2147483647) * n.ph[a] * (R(1.0) - n.ph[a]);
        sl += lam[a];
        active++;
      }
    sl /= R(active);
    R tau = tau_phi<P>(p, n.ph);
#pragma unroll
    for (int a = 0; a < P; a++)
      if (act[a]) dp[a] = p.dt * (lam[a] - sl) / (tau * p.epsilon);
  }
  // the projection also runs where no phase is active: it lifts negative phi
  project_simplex<P>(n.ph, act, dp);
}

// delta-phi of one cell  (calculate_divergence_phasefield.h:4-62)
// (T: the cell's temperature, used with NI only)
template <int P, int C, class R, bool NI = false, bool MPI = false>
__device__ __forceinline__ void cell_dphi(const DevParams<R>& p, const Nbhd<P, R>& n, const R* mu, R* dp,
                                          R T = R(0), const uint32_t* nzw = nullptr, R amp = R(0),
                                          R mnz = R(0)) {
  bool act[P];
  const bool any = cell_active<P>(p, n, act);
  const bool pairs = p.anisotropy && p.pair_sym;
  R dA[P], dG[P];
  if (any && pairs) aniso_pairs<P>(p, n, act, dA, dG);
  cell_dphi_rest<P, C, R, NI, MPI>(p, n, mu, act, any, pairs, dA, dG, dp, T, nzw, amp, mnz);
}

// ---------------------------------------------------------------- mu update

// s(phi) of the obstacle antitrapping  (calculate_fluxes_concentration.h:42-59)
template <int P, class R>
__device__ __forceinline__ R s_phi(const R* ph, int a) {
  R q = ph[a] * (R(1.0) - ph[a]);
  if (q > R(0)) return ph[a] * (R(1.0) - hphi<P>(ph, a)) / (sqrt(q));
  return R(0);
}

// D_ij of one cell  (functionD.h:1-15)
template <int P, int C, class R>
__device__ __forceinline__ void cell_D(const DevParams<R>& p, const R* ph, R (&D)[C][C]) {
#pragma unroll
  for (int i = 0; i < C; i++)
#pragma unroll
    for (int j = 0; j < C; j++) {
      R s = R(0);
#pragma unroll
      for (int b = 0; b < P; b++)
#pragma unroll
        for (int k = 0; k < C; k++) s += p.dcm[b][i][j][k] * ph[b];
      D[i][j] = s;
    }
}

// Antitrapping flux on one face between cell p (x or y) and its +1 neighbour q
// (calculate_fluxes_concentration.h:25-142).  g_p: normal gradients at the face,
// ct_p / ct_q: tangential centred gradients at p and q (the face's tangential
// gradient is their mean), phase fields, potentials and delta-phi of both cells.
// With NI, c(mu) of the two cells is taken at their temperatures T_p, T_q.
template <int P, int C, class R, bool NI = false>
__device__ __forceinline__ void face_jat(const DevParams<R>& p, const R* g_p, const R* ct_p, const R* ct_q,
                                         const R* ph_p, const R* ph_q, const R* mu_p, const R* mu_q,
                                         const R* dp_p, const R* dp_q, bool enabled, R* jat, R T_p = R(0),
                                         R T_q = R(0)) {
  constexpr int L = P - 1;
#pragma unroll
  for (int k = 0; k < C; k++) jat[k] = R(0);
  if (!enabled) return;
  R tl = R(0.5) * (ct_p[L] + ct_q[L]);
  R ngl = sqrt_nz(tl * tl + g_p[L] * g_p[L]);
#pragma unroll
  for (int a = 0; a < L; a++) {
    R t = R(0.5) * (ct_p[a] + ct_q[a]);
    R ngp = sqrt_nz(t * t + g_p[a] * g_p[a]);
    if (ngp != R(0)) {
      R s_q = R(0), s_p = R(0);
      if (p.obstacle) {
        s_q = s_phi<P>(ph_q, a);
        s_p = s_phi<P>(ph_p, a);
      }
      R sp = g_p[a] * g_p[L];
      sp += t * tl;
      if (ngl > R(0)) sp /= (ngl * ngp);
#pragma unroll
      for (int k = 0; k < C; k++) {
        R clq = c_mu_<C, NI>(p, mu_q, L, k, T_q), clp = c_mu_<C, NI>(p, mu_p, L, k, T_p);
        R csq = c_mu_<C, NI>(p, mu_q, a, k, T_q), csp = c_mu_<C, NI>(p, mu_p, a, k, T_p);
        if (!p.obstacle)
          jat[k] += p.at_coef[a][k] * fabs(sp) * p.well_at * ((clq - csq) * dp_q[a] + (clp - csp) * dp_p[a]) * g_p[a] / ngp;
        else
          jat[k] += p.at_coef[a][k] * fabs(sp) * R(0.5) * (s_q * (clq - csq) * dp_q[a] + s_p * (clp - csp) * dp_p[a]) * g_p[a] / ngp;
      }
    }
  }
}

// 1/x for the general LU solve.  The reference uses pow(x,-1) (matrix.h:121,127),
// which glibc evaluates correctly rounded for these arguments, i.e. equal to 1/x.
template <class R>
__device__ __forceinline__ R recip(R x) { return R(1.0) / x; }

// LU inverse with partial pivoting of matrix.h:50-114 (general mu solve)
template <int C, class R>
__device__ __forceinline__ void lu_inverse(R (&a)[C][C], R (&inv)[C][C]) {
  R fac[C][C], inv1[C][C];
  int tag[C];
#pragma unroll
  for (int k = 0; k < C; k++) tag[k] = k;
#pragma unroll
  for (int i = 0; i < C; i++)
#pragma unroll
    for (int j = 0; j < C; j++) fac[i][j] = R(0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    R big = fabs(a[k][k]);
    int t1 = k;
#pragma unroll
    for (int i = k + 1; i < C; i++)
      if (fabs(a[i][k]) > big) { t1 = i; big = a[i][k]; }
    if (t1 != k) {
      int ts = tag[k]; tag[k] = tag[t1]; tag[t1] = ts;
#pragma unroll
      for (int i = 0; i < C; i++) {
#pragma unroll
        for (int r = k + 1; r < C; r++)
          if (r == t1) { R s = a[k][i]; a[k][i] = a[r][i]; a[r][i] = s; }
      }
#pragma unroll
      for (int i = 0; i < k; i++) {
#pragma unroll
        for (int r = k + 1; r < C; r++)
          if (r == t1) { R s = fac[k][i]; fac[k][i] = fac[r][i]; fac[r][i] = s; }
      }
    }
#pragma unroll
    for (int i = k + 1; i < C; i++) {
      R f = -a[i][k] / a[k][k];
      fac[i][k] = -f;
#pragma unroll
      for (int j = k; j < C; j++) a[i][j] = f * a[k][j] + a[i][j];
    }
  }
#pragma unroll
  for (int col = 0; col < C; col++) {
    R v1[C], v[C];
    v1[0] = (col == 0) ? R(1.0) : R(0);
#pragma unroll
    for (int i = 1; i < C; i++) {
      R s = R(0);
#pragma unroll
      for (int j = 0; j < i; j++) s = s - fac[i][j] * v1[j];
      v1[i] = ((i == col) ? R(1.0) : R(0)) + s;
    }
    v[C - 1] = v1[C - 1] * recip(a[C - 1][C - 1]);
#pragma unroll
    for (int i = C - 2; i >= 0; i--) {
      R s = R(0);
#pragma unroll
      for (int j = i + 1; j < C; j++) s = s - a[i][j] * v[j];
      v[i] = (v1[i] + s) * recip(a[i][i]);
    }
#pragma unroll
    for (int j = 0; j < C; j++) inv1[j][col] = v[j];
  }
#pragma unroll
  for (int j = 0; j < C; j++)
#pragma unroll
    for (int q = 0; q < C; q++)
#pragma unroll
      for (int t = 0; t < C; t++)
        if (tag[j] == t) inv[q][t] = inv1[q][j];
}

// mu and phi update of one cell from its face fluxes
// (calculate_divergence_concentration.h:4-153).  jat*/Dm*/gm*: antitrapping flux,
// face mobility and mu gradient on the faces front (x|x+1), back (x-1|x),
// right (y|y+1), left (y-1|y).
template <int P, int C, class R, bool NI = false, class Pm>
__device__ __forceinline__ void cell_update(const Pm& p, const R* ph, const R* mu, const R* dp,
                                            const R* jf, const R* jb, const R* jr, const R* jl,
                                            const R (&Dmf)[C][C], const R (&Dmb)[C][C],
                                            const R (&Dmr)[C][C], const R (&Dml)[C][C],
                                            const R* gmf, const R* gmb, const R* gmr, const R* gml,
                                            R* ph_o, R* mu_o, R* dmu, R T = R(0), R* cst = nullptr) {
  R divflux[C], divjat[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    divflux[k] = R(0);
#pragma unroll
    for (int l = 0; l < C; l++) {
      divflux[k] += div_dx(Dmf[k][l] * gmf[l] - Dmb[k][l] * gmb[l], p);
      divflux[k] += div_dy(Dmr[k][l] * gmr[l] - Dml[k][l] * gml[l], p);
    }
    divjat[k] = div_dx((jf[k] - jb[k]) * p.jscale, p);
    divjat[k] += div_dy((jr[k] - jl[k]) * p.jscale, p);
  }
  int bulk = -1;
#pragma unroll
  for (int a = P - 1; a >= 0; a--)
    if (ph[a] == R(1.0)) bulk = a;
  if (cst) {
    // composition field (MPI calculate_divergence_concentration.h:438-470):
    // every cell adds dt div(M grad mu) - div(j_at) to c; a bulk cell then
    // takes mu = Mu_a(c), an interface cell keeps the update below
#pragma unroll
    for (int k = 0; k < C; k++) cst[k] += p.dt * (divflux[k]) - divjat[k];
  }
  if (bulk >= 0 && cst) {
#pragma unroll
    for (int a = 0; a < P; a++)
      if (a == bulk) {
#pragma unroll
        for (int k = 0; k < C; k++) {
          mu_o[k] = Mu_of_c_<C, NI>(p, cst, a, k, T);
          dmu[k] = mu_o[k] - mu[k];
        }
      }
  } else if (bulk >= 0) {
    R cn[C], dcb[C];
#pragma unroll
    for (int k = 0; k < C; k++) dcb[k] = p.dt * (divflux[k]) - divjat[k];
#pragma unroll
    for (int a = 0; a < P; a++)
      if (a == bulk) {
#pragma unroll
        for (int k = 0; k < C; k++) cn[k] = c_mu_<C, NI>(p, mu, a, k, T) + p.dt * (divflux[k]) - divjat[k];
#pragma unroll
        for (int k = 0; k < C; k++) {
          mu_o[k] = Mu_of_c_<C, NI>(p, cn, a, k, T);
          // the same update as an increment of the linear map Mu(c): dMu/dc . delta_c
          R d = R(0);
#pragma unroll
          for (int j = 0; j < C; j++) d += (j == k ? R(2.0) * p.A[a][k][k] : p.A[a][k][j]) * dcb[j];
          dmu[k] = d;
        }
      }
  } else {
    R sum[C], dc[C], dcdmu[C][C], h[P];
#pragma unroll
    for (int k = 0; k < C; k++) sum[k] = R(0);
#pragma unroll
    for (int a = 0; a < P; a++) {
      R sdh = R(0);
#pragma unroll
      for (int b = 0; b < P; b++) sdh += dhphi<P>(ph, a, b) * dp[b];
#pragma unroll
      for (int k = 0; k < C; k++) sum[k] += c_mu_<C, NI>(p, mu, a, k, T) * sdh;
      h[a] = hphi<P>(ph, a);
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      if constexpr (NI) {
        // dcbdT_phase is allocated zero and never set, nor is the GRADIENT member
        // of temperature_gradientY, so the term is a signed zero
        // (calculate_divergence_concentration.h:22-40,85)
        R sdc = R(0);
#pragma unroll
        for (int a = 0; a < P; a++) sdc += R(0) * h[a];
        const R gm = R(0);
        dc[k] = p.dt * (divflux[k]) - divjat[k] - sum[k] - sdc * p.dt * (-gm * p.tgv);
      } else {
        dc[k] = p.dt * (divflux[k]) - divjat[k] - sum[k];
      }
#pragma unroll
      for (int l = 0; l < C; l++) {
        dcdmu[k][l] = R(0);
#pragma unroll
        for (int a = 0; a < P; a++) dcdmu[k][l] += p.cmu[a][k][l] * h[a];
      }
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      mu_o[k] = mu[k];
      dmu[k] = R(0);
    }
    if (p.mu_solver == GP_MU_BINARY) {
      R inv = R(1.0) / dcdmu[0][0];
      dmu[0] = dc[0] * inv;
      mu_o[0] = mu[0] + dmu[0];
    } else if (C == 2 && p.mu_solver == GP_MU_TERNARY) {
      R DET = dcdmu[0][0] * dcdmu[C - 1][C - 1] - dcdmu[0][C - 1] * dcdmu[C - 1][0];
      R i00 = dcdmu[C - 1][C - 1] / DET, i11 = dcdmu[0][0] / DET;
      R i01 = -dcdmu[0][C - 1] / DET, i10 = -dcdmu[C - 1][0] / DET;
      R d0 = R(0), d1 = R(0);
      d0 += i00 * dc[0];
      d0 += i01 * dc[C - 1];
      d1 += i10 * dc[0];
      d1 += i11 * dc[C - 1];
      dmu[0] = d0;
      dmu[C - 1] = d1;
      mu_o[0] = d0 + mu[0];
      mu_o[C - 1] = d1 + mu[C - 1];
    } else if (p.mu_solver == GP_MU_DILUTE) {
#pragma unroll
      for (int k = 0; k < C; k++) {
        R inv = R(1.0) / dcdmu[k][k];
        dmu[k] = dc[k] * inv;
        mu_o[k] = mu[k] + dmu[k];
      }
    } else {
      R inv[C][C];
      lu_inverse<C>(dcdmu, inv);
#pragma unroll
      for (int k = 0; k < C; k++) {
        R s = R(0);
#pragma unroll
        for (int l = 0; l < C; l++) s = s + inv[k][l] * dc[l];
        dmu[k] = s;
        mu_o[k] = s + mu[k];
      }
    }
  }
#pragma unroll
  for (int b = 0; b < P; b++) ph_o[b] = ph[b] + dp[b];
}

// ---------------------------------------------------------------- smoothing

// Pre-loop smoothing sweep (NSMOOTH > 1): smooth() of solverloop/solverloop.h:72-90.
// delta-phi without the driving force, isotropic gradient sums also for
// anisotropic runs (function_A_01.h:73-99,220-262 return 2*(sum1 + sum2) with
// sum2 = 0; function_A_00.h returns 2*sum), obstacle/well terms without sign
// tests (functionW_01.h:41-63, functionW_02.h:35-58), unweighted projection
// (simplex_projection.h:50-90).
template <int P, class R>
__device__ __forceinline__ R dwdphi_smooth(const DevParams<R>& p, const R* ph, const bool* act, int a) {
  R sum = R(0);
#pragma unroll
  for (int b = 0; b < P; b++)
    if (b != a && act[b]) {
      if (p.obstacle) sum += p.gamma[a][b] * ph[b];
      else sum += R(2.0) * p.gamma[a][b] * (ph[b] * ph[b] * ph[a]);
    }
  sum *= p.w_pref;
#pragma unroll
  for (int b = 0; b < P; b++)
#pragma unroll
    for (int c = 0; c < P; c++)
      if (b != a && c != a && b < c && act[b] && act[c]) sum += p.gamma_abc[a][b][c] * ph[b] * ph[c];
  return sum;
}

template <int P, class R>
__device__ __forceinline__ void project_unweighted(const R* ph, const bool* act, R* dp) {
  int count = 0;
#pragma unroll
  for (int a = 0; a < P; a++)
    if (act[a] && (ph[a] + dp[a]) > R(0) && (ph[a] + dp[a]) < R(1.0)) count++;
  bool done = false;
#pragma unroll
  for (int a = 0; a < P; a++) {
    if (done || !act[a]) continue;
    if ((ph[a] + dp[a]) > R(1.0)) {
      dp[a] = (R(1.0) - ph[a]);
#pragma unroll
      for (int b = 0; b < P; b++)
        if (act[b] && b != a) dp[b] = -ph[b];
      done = true;
      continue;
    }
    if ((ph[a] + dp[a]) < R(0)) {
      R D = fabs(dp[a] + ph[a]);
      dp[a] += D;
#pragma unroll
      for (int b = 0; b < P; b++)
        if (act[b] && b != a && (ph[b] + dp[b]) > R(0) && (ph[b] + dp[b]) < R(1.0)) dp[b] -= D / R(count);
    }
  }
}

template <int P, int C, class R>
__device__ __forceinline__ void cell_dphi_smooth(const DevParams<R>& p, const Nbhd<P, R>& n, R* dp) {
  R divphi[P], lam[P];
  bool act[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    divphi[a] = div_dx(n.gXc[a] - n.gXb[a], p);
    divphi[a] += div_dy(n.gYc[a] - n.gYl[a], p);
    act[a] = fabs(divphi[a]) > R(0);
    dp[a] = R(0);
  }
  R sl = R(0), active = R(0);
#pragma unroll
  for (int a = 0; a < P; a++)
    if (act[a]) {
      R dA = R(0), dv = R(0);
#pragma unroll
      for (int b = 0; b < P; b++) {
        if (b == a || !n.present[b]) continue;  // an absent phase contributes exact zeros
        R sp = R(0);
        sp += (n.ph[a] * n.cXc[b] - n.ph[b] * n.cXc[a]) * n.cXc[b];
        sp += (n.ph[a] * n.cYc[b] - n.ph[b] * n.cYc[a]) * n.cYc[b];
        sp *= p.gamma[a][b];
        dA += sp;
        R fc = n.sXc[a] * n.gXc[b] - n.sXc[b] * n.gXc[a];
        R fb = n.sXb[a] * n.gXb[b] - n.sXb[b] * n.gXb[a];
        R d1 = div_dx(fc * (-n.sXc[b]) - (fb * (-n.sXb[b])), p);
        R gc = n.sYc[a] * n.gYc[b] - n.sYc[b] * n.gYc[a];
        R gl = n.sYl[a] * n.gYl[b] - n.sYl[b] * n.gYl[a];
        d1 += div_dy(gc * (-n.sYc[b]) - (gl * (-n.sYl[b])), p);
        d1 *= p.gamma[a][b];
        dv += d1;
      }
      const R A = p.anisotropy ? R(2.0) * (dA + R(0)) : R(2.0) * dA;
      const R D = p.anisotropy ? R(2.0) * (dv + R(0)) : R(2.0) * dv;
      lam[a] = p.epsilon * (-A + D) - p.inv_eps * dwdphi_smooth<P>(p, n.ph, act, a);
      sl += lam[a];
      active += R(1);
    }
  if (active != R(0)) {
    sl /= active;
    R tau = tau_phi<P>(p, n.ph);
#pragma unroll
    for (int a = 0; a < P; a++)
      if (act[a]) dp[a] = p.dt * (lam[a] - sl) / (tau * p.epsilon);
  }
  project_unweighted<P>(n.ph, act, dp);
}

// mu update of the smoothing sweep: diffusion alone, general LU inverse for any
// solver flag, mu + delta_mu (calculate_divergence_concentration.h:154-253)
template <int P, int C, class R>
__device__ __forceinline__ void cell_update_smooth(const DevParams<R>& p, const R* ph, const R* mu,
                                                   const R (&Dmf)[C][C], const R (&Dmb)[C][C],
                                                   const R (&Dmr)[C][C], const R (&Dml)[C][C],
                                                   const R* gmf, const R* gmb, const R* gmr, const R* gml,
                                                   R* mu_o, R* dmu) {
  R divflux[C];
#pragma unroll
  for (int k = 0; k < C; k++) {
    divflux[k] = R(0);
#pragma unroll
    for (int l = 0; l < C; l++) {
      divflux[k] += div_dx(Dmf[k][l] * gmf[l] - Dmb[k][l] * gmb[l], p);
      divflux[k] += div_dy(Dmr[k][l] * gmr[l] - Dml[k][l] * gml[l], p);
    }
  }
  int bulk = -1;
#pragma unroll
  for (int a = P - 1; a >= 0; a--)
    if (ph[a] == R(1.0)) bulk = a;
  if (bulk >= 0) {
    R cn[C];
#pragma unroll
    for (int a = 0; a < P; a++)
      if (a == bulk) {
#pragma unroll
        for (int k = 0; k < C; k++) cn[k] = c_mu<C>(p, mu, a, k) + p.dt * (divflux[k]);
#pragma unroll
        for (int k = 0; k < C; k++) {
          mu_o[k] = Mu_of_c<C>(p, cn, a, k);
          R d = R(0);
#pragma unroll
          for (int j = 0; j < C; j++) d += (j == k ? R(2.0) * p.A[a][k][k] : p.A[a][k][j]) * (p.dt * divflux[j]);
          dmu[k] = d;
        }
      }
  } else {
    R dc[C], dcdmu[C][C], h[P], inv[C][C];
#pragma unroll
    for (int a = 0; a < P; a++) h[a] = hphi<P>(ph, a);
#pragma unroll
    for (int k = 0; k < C; k++) {
      dc[k] = p.dt * (divflux[k]);
#pragma unroll
      for (int l = 0; l < C; l++) {
        dcdmu[k][l] = R(0);
#pragma unroll
        for (int a = 0; a < P; a++) dcdmu[k][l] += p.cmu[a][k][l] * h[a];
      }
    }
    lu_inverse<C>(dcdmu, inv);
#pragma unroll
    for (int k = 0; k < C; k++) {
      R s = R(0);
#pragma unroll
      for (int l = 0; l < C; l++) s = s + inv[k][l] * dc[l];
      dmu[k] = s;
      mu_o[k] = s + mu[k];
    }
  }
}

}  // namespace GPK_NS
