// gp_step.hip -- C ABI of the MI355X grand-potential 2-D step (include/gpstep.h).
//
// Context creation copies the host-derived constant tables into a device
// DevParams<R> block, allocates the padded field planes, and dispatches each
// call to the kernels instantiated for the context's (P, C, real type).
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>
#include <new>

#include "gp_ctx.hpp"
#include "gp_kernels.hpp"
#include "gpio.h"

// (P, C) pairs with compiled kernels; other combinations are rejected with
// GP_E_UNSUPPORTED.  Must match the GP_INSTANTIATE lines of gp_inst_p*.hip.
#define GP_PC_LIST(X) \
  X(2, 1) X(3, 1) X(4, 1) X(5, 1) X(6, 1) X(7, 1) X(8, 1) X(9, 1) \
  X(2, 2) X(3, 2) X(4, 2) X(5, 2) X(6, 2) X(2, 3) X(3, 3) X(4, 3)

static bool pc_supported(int P, int C) {
#define GP_PC_TEST(P_, C_) if (P == P_ && C == C_) return true;
  GP_PC_LIST(GP_PC_TEST)
#undef GP_PC_TEST
  return false;
}

template <class R>
static void fill_devparams(const gp_params &h, int rx, int ry, int pitch, long plane, gpk::DevParams<R> &d) {
  memset(&d, 0, sizeof(d));
  const int P = h.nphases, C = h.ncomp, L = P - 1;
  d.plane = plane;
  d.rx = rx;
  d.ry = ry;
  d.pitch = pitch;
  d.mesh_x = (int)h.mesh_x;
  d.mesh_y = (int)h.mesh_y;
  d.obstacle = h.obstacle;
  d.anisotropy = h.anisotropy;
  d.mu_solver = h.mu_solver;
  d.yskip = (h.mpi & GP_MPI_YSKIP) ? (int)h.mesh_y + 4 : (int)h.mesh_y - 2;
  {
    int e;
    d.pow2_dx = frexp(h.dx, &e) == 0.5;
    d.pow2_dy = frexp(h.dy, &e) == 0.5;
  }
  for (int f = 0; f < 2; f++) {
    // slots 0,1,2 = ghosts 0,1,2 (faces X- / Y-), slots 3,4,5 = ghosts n-3, n-2, n-1 (X+ / Y+)
    d.gsrc[f][0][0] = (int)h.bc_proxy[f][GP_FACE_XMIN][2];
    d.gsrc[f][0][1] = (int)h.bc_proxy[f][GP_FACE_XMIN][1];
    d.gsrc[f][0][2] = (int)h.bc_proxy[f][GP_FACE_XMIN][0];
    d.gsrc[f][0][3] = (int)h.bc_proxy[f][GP_FACE_XMAX][0];
    d.gsrc[f][0][4] = (int)h.bc_proxy[f][GP_FACE_XMAX][1];
    d.gsrc[f][0][5] = (int)h.bc_proxy[f][GP_FACE_XMAX][2];
    d.gsrc[f][1][0] = (int)h.bc_proxy[f][GP_FACE_YMIN][2];
    d.gsrc[f][1][1] = (int)h.bc_proxy[f][GP_FACE_YMIN][1];
    d.gsrc[f][1][2] = (int)h.bc_proxy[f][GP_FACE_YMIN][0];
    d.gsrc[f][1][3] = (int)h.bc_proxy[f][GP_FACE_YMAX][0];
    d.gsrc[f][1][4] = (int)h.bc_proxy[f][GP_FACE_YMAX][1];
    d.gsrc[f][1][5] = (int)h.bc_proxy[f][GP_FACE_YMAX][2];
    for (int ax = 0; ax < 2; ax++) {  // the band between the sources of the low and the high ghosts
      const int n = ax ? d.ry : d.rx;
      int lo = 0, hi = n - 1;
      for (int s = 0; s < 6; s++) {
        const int g = d.gsrc[f][ax][s];
        if (g < 0) continue;
        if (2 * g <= n) lo = std::max(lo, g + 1);
        else hi = std::min(hi, g - 1);
      }
      d.gfree[f][ax][0] = lo;
      d.gfree[f][ax][1] = hi;
    }
  }
  // scalar constants, each formed in binary64 as the reference forms it
  d.dx = (R)h.dx;
  d.dy = (R)h.dy;
  d.dt = (R)h.dt;
  d.two_dy = (R)(2.0 * h.dy);
  d.inv_dx = (R)(1.0 / h.dx);
  d.inv_dy = (R)(1.0 / h.dy);
  d.inv_two_dy = (R)(1.0 / (2.0 * h.dy));
  d.epsilon = (R)h.epsilon;
  d.inv_eps = (R)(1.0 / h.epsilon);
  d.tau = (R)h.tau;
  d.w_pref = (R)(h.obstacle ? 16.0 / (M_PI * M_PI) : 9.0);
  d.jscale = (R)(h.obstacle ? (-0.25 * M_PI * h.epsilon) : (-1.0 * h.epsilon));
  d.well_at = (R)(0.5 / sqrt(2.0));
  d.diff_s = (R)h.diffusivity[0][0][0];
  d.diff_l = (R)h.diffusivity[h.nphases - 1][0][0];
  d.pair_sym = 1;
  for (int a = 0; a < P; a++)
    for (int b = 0; b < P; b++) {
      if (h.dab[a][b] != h.dab[b][a]) d.pair_sym = 0;
      for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++)
          if (h.rot[a][b][i][j] != h.rot[b][a][i][j] || h.rot_inv[a][b][i][j] != h.rot_inv[b][a][i][j]) d.pair_sym = 0;
    }
  for (int a = 0; a < P; a++) {
    for (int b = 0; b < P; b++) {
      d.gamma[a][b] = (R)h.gamma[a][b];
      d.tau_ab[a][b] = (R)h.tau_ab[a][b];
      d.dab[a][b] = (R)h.dab[a][b];
      for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) {
          d.rot[a][b][i][j] = (R)h.rot[a][b][i][j];
          d.rot_inv[a][b][i][j] = (R)h.rot_inv[a][b][i][j];
        }
      for (int c = 0; c < P; c++) d.gamma_abc[a][b][c] = (R)h.gamma_abc[a][b][c];
    }
    for (int k = 0; k < C; k++) {
      d.at_coef[a][k] = (R)(a < L ? (1.0 - h.diffusivity[a][k][k] / h.diffusivity[L][k][k]) : 0.0);
      d.Bsh[a][k] = (R)(h.Beq[a][k] + h.dBbdT[a][k] * (h.T - h.Teq));
      d.B[a][k] = (R)h.B[a][k];
      for (int l = 0; l < C; l++) {
        d.A[a][k][l] = (R)h.A[a][k][l];
        d.cmu[a][k][l] = (R)h.cmu[a][k][l];
        for (int m = 0; m < C; m++) d.dcm[a][k][l][m] = (R)(h.diffusivity[a][k][m] * h.cmu[a][m][l]);
      }
    }
    d.Cf[a] = (R)h.Cf[a];
  }
  // the mobility of a cell one-hot in phase a and the mean of two such cells,
  // with the operations of cell_D and bulk_mu_v in their order (each term
  // dcm * 1 or dcm * 0, exact; no contraction in this file), so that the
  // light mu sweeps may read it instead of forming it
  for (int a = 0; a < P; a++)
    for (int i = 0; i < C; i++)
      for (int j = 0; j < C; j++) {
        R s = R(0);
        for (int b = 0; b < P; b++)
          for (int k = 0; k < C; k++) s += d.dcm[b][i][j][k] * (b == a ? R(1.0) : R(0));
        d.Dm_bulk[a][i][j] = (s + s) * R(0.5);
      }
  // non-isothermal runs
  d.ni = !h.isothermal;
  d.Teq = (R)h.Teq;
  d.tgG = (R)(h.isothermal ? 0.0 : (h.tempgrad[1]) * h.dy / (h.tempgrad[2]));
  d.tgv = (R)h.tempgrad[4];
  for (int a = 0; a < P; a++)
    for (int k = 0; k < C; k++) {
      d.Beq[a][k] = (R)h.Beq[a][k];
      d.dBbdT[a][k] = (R)h.dBbdT[a][k];
      d.dC[a][k] = (R)h.delta_C[a][k];
      d.ceqL[a][k] = (R)h.ceq[a][L][k];
      d.ceqS[a][k] = (R)h.ceq[a][a][k];
    }
  for (int a = 0; a < P; a++) {
    d.dTs[a] = (R)h.delta_T_s[a];
    d.dTl[a] = (R)h.delta_T_l[a];
  }
  // MPI solver semantics
  d.mpi = h.mpi;
  d.V = (R)h.V;
  d.noise4amp = (R)(4.0 * h.amp_noise);
  d.mpi_noise = (h.mpi & GP_MPI_NOISE) && h.noise;
  {
    // drand48's map x -> a x + c (mod 2^48) applied 2^k times, and applied once
    // per draw of a step's phase sweep ((rows_x-2)(rows_y-2) draws)
    const unsigned long long M = gpk::kLcgMask;
    unsigned long long A = 0x5DEECE66DULL, Cc = 0xBULL;
    for (int k = 0; k < 34; k++) {
      d.lcg[k][0] = A;
      d.lcg[k][1] = Cc;
      Cc = (A * Cc + Cc) & M;
      A = (A * A) & M;
    }
    const unsigned long long n = (unsigned long long)(rx - 2) * (unsigned long long)(ry - 2);
    unsigned long long SA = 1, SC = 0;
    for (int k = 0; k < 34; k++)
      if ((n >> k) & 1ull) {
        SC = (d.lcg[k][0] * SC + d.lcg[k][1]) & M;
        SA = (d.lcg[k][0] * SA) & M;
      }
    d.lcg_step[0] = SA;
    d.lcg_step[1] = SC;
  }
  // temperature ghost rows (y faces): rows 0,1,2 copy proxies 2,1,0 of Y-, rows
  // ry-3.. copy proxies 0,1,2 of Y+ (boundary_serial.h:120-175); other types copy nothing
  for (int j = 0; j < 6; j++) d.tsrc[j] = -1;
  {
    const int tl = h.bc_type_T[GP_FACE_YMIN], th = h.bc_type_T[GP_FACE_YMAX];
    if (tl == GP_BC_NEUMANN || tl == GP_BC_PERIODIC)
      for (int j = 0; j < 3; j++) d.tsrc[j] = (int)h.bc_proxy_T[GP_FACE_YMIN][2 - j];
    if (th == GP_BC_NEUMANN || th == GP_BC_PERIODIC)
      for (int j = 0; j < 3; j++) d.tsrc[3 + j] = (int)h.bc_proxy_T[GP_FACE_YMAX][j];
  }
}

template <class R, class S>
static int load_state(gp_ctx *c, const S *dphi_src, const S *dmu_src) {
  const gpk::DevParams<R> *prm = (const gpk::DevParams<R> *)c->dprm;
  dim3 blk(gpk::BX, gpk::BY), g((c->hp.mesh_y + gpk::BX - 1) / gpk::BX, (c->hp.mesh_x + gpk::BY - 1) / gpk::BY);
  dim3 gi((c->hp.mesh_y + gpk::BX - 1) / gpk::BX, (c->hp.mesh_x + gpk::BY - 1) / gpk::BY);
  hipLaunchKernelGGL((gpk::k_pack<R, S>), g, blk, 0, c->stream, prm, dphi_src, (R *)c->phi[c->cur], c->P);
  hipLaunchKernelGGL((gpk::k_pack<R, S>), g, blk, 0, c->stream, prm, dmu_src, (R *)c->mu[c->cur], c->C);
  hipLaunchKernelGGL((gpk::k_ghosts<R>), gi, blk, 0, c->stream, prm, (R *)c->phi[c->cur], (R *)c->mu[c->cur], c->P, c->C);
  if (c->mulo[c->cur]) GP_HIP_CHECK(hipMemsetAsync(c->mulo[c->cur], 0, (size_t)c->plane * c->esize * c->C, c->stream));
  GP_HIP_CHECK(hipGetLastError());
  c->flags_valid = 0;
  c->oh_valid = 0;
  c->stepped = 0;
  c->tstep = 0;
  c->shift_off = 0;
  c->shift_pend = 0;
  return GP_OK;
}

// Ghost images of the composition planes (mu's copies), binary64 contexts.
static hipError_t comp_ghosts(gp_ctx *c) {
  dim3 blk(gpk::BX, gpk::BY), gi((c->hp.mesh_y + gpk::BX - 1) / gpk::BX, (c->hp.mesh_x + gpk::BY - 1) / gpk::BY);
  hipLaunchKernelGGL((gpk::k_ghosts<double>), gi, blk, 0, c->stream, (const gpk::DevParams<double> *)c->dprm,
                     (double *)c->dcomp, (double *)c->dcomp, 0, c->C);
  return hipGetLastError();
}

// Composition planes from the current fields (sum_a h_a c_a(mu) per cell).
static int comp_init(gp_ctx *c) {
  int rc = GP_E_UNSUPPORTED;
#define GP_DISPATCH_COMP(P_, C_) \
  if (c->P == P_ && c->C == C_) rc = gpk::run_comp_init<P_, C_, double>(c);
  GP_PC_LIST(GP_DISPATCH_COMP)
#undef GP_DISPATCH_COMP
  return rc;
}

template <class R, class S>
static int store_state(gp_ctx *c, S *dphi_dst, S *dmu_dst) {
  const gpk::DevParams<R> *prm = (const gpk::DevParams<R> *)c->dprm;
  dim3 blk(gpk::BX, gpk::BY), g((c->hp.mesh_y + gpk::BX - 1) / gpk::BX, (c->hp.mesh_x + gpk::BY - 1) / gpk::BY);
  hipLaunchKernelGGL((gpk::k_unpack<R, S>), g, blk, 0, c->stream, prm, (const R *)c->phi[c->cur], dphi_dst, c->P);
  hipLaunchKernelGGL((gpk::k_unpack<R, S>), g, blk, 0, c->stream, prm, (const R *)c->mu[c->cur], dmu_dst, c->C);
  GP_HIP_CHECK(hipGetLastError());
  return GP_OK;
}

// Bytes of a grid's fields in transit from and to host memory (P + C unpadded
// binary64 planes).
static size_t transit_bytes(const gp_ctx *c) {
  return sizeof(double) * (size_t)c->hp.mesh_x * c->hp.mesh_y * (c->P + c->C);
}

// Device buffer for them, for the length of one call: the caller's work on it
// has finished when it goes out of scope.  A grid that needs at most
// GP_TRANSIT_KEEP bytes uses a buffer that its context keeps (the members of an
// ensemble share the ensemble's), allocated on first use and used by one call at
// a time; for a larger one it is allocated and given back by the call.  Keeping
// it pays in this range and is small beside the fields: set_state + get_state of
// a context took 475 us with and 400 us without hipMalloc and hipFree at 3.4 MiB,
// 716 and 632 at 6 MiB, but 1237 and 1169 at 12 MiB, 2448 and 2390 at 24 MiB
// (and the same at 1.5 MiB, where the runtime hands out parts of a chunk that it
// holds); an adjoint pass of 200 steps at 512^2 took 15.55 and 15.27 ms.
struct Transit {
  double *d = nullptr;  // null: no memory
  explicit Transit(gp_ctx *c) {
    gp_ctx *m = c->stage_of;
    if (transit_bytes(c) <= m->stage_bytes) {
      hold = std::unique_lock<std::mutex>(m->stage_mu);
      if (!m->stage) m->stage = alloc(m->stage_bytes);
      if ((d = m->stage)) return;
      hold.unlock();
    }
    d = own = alloc(transit_bytes(c));
  }
  ~Transit() {
    if (own) (void)hipFree(own);
  }
  Transit(const Transit &) = delete;
  Transit &operator=(const Transit &) = delete;

 private:
  double *own = nullptr;
  std::unique_lock<std::mutex> hold;
  static double *alloc(size_t bytes) {
    double *p = nullptr;
    if (hipMalloc((void **)&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
  }
};

extern "C" {

const char *gp_strerror(int code) {
  switch (code) {
    case GP_OK: return "ok";
    case GP_E_ARG: return "invalid argument or parameters";
    case GP_E_UNSUPPORTED: return "valid input not supported by this build";
    case GP_E_HIP: return "HIP runtime error";
    case GP_E_NOMEM: return "allocation failed";
    case GP_E_NONFINITE: return "non-finite values in the fields";
    case GP_E_IO: return "file not found or unreadable";
    case GP_E_NODEVICE: return "no HIP device";
    case GP_E_SCRATCH: return "grid too large for the no-allocation scratch array (gp_step_noalloc)";
    default: return "unknown error";
  }
}

// ------------------------------------------------------- phase-field noise

// glibc rand() (random() of type 3) as the lagged-Fibonacci state the noise
// kernels advance: after srand(seed) (x_0 = seed, x_i = 16807 x_{i-1} mod
// 2^31-1 by Schrage's method for i < 31, then x_n = x_{n-31} + x_{n-3} mod
// 2^32 with 310 values discarded), the last 31 words, oldest first.
static void noise_seed_state(unsigned seed, uint32_t st[31]) {
  uint32_t r[31];
  int32_t word = seed ? (int32_t)seed : 1;
  r[0] = (uint32_t)word;
  for (int i = 1; i < 31; i++) {
    const int32_t hi = word / 127773, lo = word % 127773;
    word = 16807 * lo - 2836 * hi;
    if (word < 0) word += 2147483647;
    r[i] = (uint32_t)word;
  }
  // ring of 31 words; the oldest sits at f, x_{n-3} at f + 28 (mod 31)
  int f = 3;
  for (int k = 0; k < 310; k++) {
    const int b = f + 28 >= 31 ? f - 3 : f + 28;
    r[f] += r[b];
    f = f + 1 == 31 ? 0 : f + 1;
  }
  for (int i = 0; i < 31; i++) st[i] = r[(f + i) % 31];
}

// M^(256 * 2^k) (mod 2^32) for k < 24, row-major 31 x 31: M advances the state
// (x_{n-31} .. x_{n-1}) by one word.
static void noise_jump_tables(std::vector<uint32_t> &out) {
  constexpr int N = 31;
  auto mul = [](const std::vector<uint32_t> &A, const std::vector<uint32_t> &B) {
    std::vector<uint32_t> Cm(N * N, 0u);
    for (int i = 0; i < N; i++)
      for (int k = 0; k < N; k++) {
        const uint32_t a = A[i * N + k];
        if (!a) continue;
        for (int j = 0; j < N; j++) Cm[i * N + j] += a * B[k * N + j];
      }
    return Cm;
  };
  std::vector<uint32_t> M(N * N, 0u);
  for (int i = 0; i + 1 < N; i++) M[i * N + i + 1] = 1u;  // shift
  M[(N - 1) * N + 0] = 1u;                                // x_n = x_{n-31}
  M[(N - 1) * N + 28] += 1u;                              //     + x_{n-3}
  std::vector<uint32_t> P = M;
  for (int k = 0; k < 8; k++) P = mul(P, P);  // M^256
  out.clear();
  for (int k = 0; k < 24; k++) {
    out.insert(out.end(), P.begin(), P.end());
    P = mul(P, P);
  }
}

// Releases a context: its queued work finishes first, then the captured step
// blocks (which name its buffers) are destroyed, then the buffers are freed.
static void release_graphs(gp_ctx *c) {
  for (int g = 0; g < GP_GRAPH_SLOTS; g++)
    for (int i = 0; i < 2; i++)
      if (c->gcache[g][i]) (void)hipGraphExecDestroy(c->gcache[g][i]), c->gcache[g][i] = nullptr;
}

static void free_ctx(gp_ctx *c) {
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  release_graphs(c);
  for (int i = 0; i < 2; i++) {
    if (c->phi[i]) (void)hipFree(c->phi[i]);
    if (c->mu[i]) (void)hipFree(c->mu[i]);
    if (c->mulo[i]) (void)hipFree(c->mulo[i]);
  }
  if (c->dphi) (void)hipFree(c->dphi);
  if (c->stage) (void)hipFree(c->stage);
  if (c->dcode) (void)hipFree(c->dcode);
  if (c->dsplit) (void)hipFree(c->dsplit);
  if (c->dcells) (void)hipFree(c->dcells);
  if (c->doh) (void)hipFree(c->doh);
  if (c->dcells6) (void)hipFree(c->dcells6);
  if (c->dcomp) (void)hipFree(c->dcomp);
  if (c->drstate) (void)hipFree(c->drstate);
  for (void *b : {(void *)c->dnz_state, (void *)c->dnz_jump, (void *)c->dnz_raw, (void *)c->dnz_off,
                  (void *)c->dnz_rows, (void *)c->dnz_total})
    if (b) (void)hipFree(b);
  if (c->dprm) (void)hipFree(c->dprm);
  if (c->dpart) (void)hipFree(c->dpart);
  if (c->drow) (void)hipFree(c->drow);
  for (int i = 0; i < 2; i++)
    if (c->dflag[i]) (void)hipFree(c->dflag[i]);
  if (c->ddeps) (void)hipFree(c->ddeps);
  if (c->dlist) (void)hipFree(c->dlist);
  if (c->dlist_all) (void)hipFree(c->dlist_all);
  if (c->dcnt) (void)hipFree(c->dcnt);
  if (c->dinst) (void)hipFree(c->dinst);
  if (c->dtinst) (void)hipFree(c->dtinst);
  if (c->own_stream) (void)hipStreamDestroy(c->own_stream);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  delete c;
}

// A context with its fields; own_stream: create a stream of its own (ensemble
// members enqueue on their master's stream instead).
static int ctx_create(const gp_params *p, int dtype, bool own_stream, gp_ctx **out) {
  if (!p || !out || (dtype != GP_F64 && dtype != GP_F32)) return GP_E_ARG;
  *out = nullptr;
  char err[200];
  int rc = gp_check_supported(p, err, sizeof err);
  if (rc) return rc;
  if (!pc_supported(p->nphases, p->ncomp)) return GP_E_UNSUPPORTED;
  // the MPI solver's semantics: binary64, isothermal, its own noise only
  if (p->mpi & ~GP_MPI_ALL) return GP_E_ARG;
  if (p->mpi && (dtype != GP_F64 || !p->isothermal || (p->noise && !(p->mpi & GP_MPI_NOISE)))) return GP_E_UNSUPPORTED;
  if ((p->mpi & (GP_MPI_DPSI_V | GP_MPI_NOISE | GP_MPI_TAU)) && !(p->V > 0.0)) return GP_E_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return GP_E_NODEVICE;
  gp_ctx *c = new (std::nothrow) gp_ctx();
  if (!c) return GP_E_NOMEM;
  c->hp = *p;
  c->dtype = dtype;
  c->P = p->nphases;
  c->C = p->ncomp;
  c->rx = (int)p->mesh_x + 6;
  c->ry = (int)p->mesh_y + 6;
  c->esize = dtype == GP_F64 ? 8 : 4;
  c->stage_of = c;
  c->stage_bytes = transit_bytes(c) <= GP_TRANSIT_KEEP ? transit_bytes(c) : 0;
  int align = (int)(256 / c->esize);
  c->pitch = (c->ry + align - 1) / align * align;
  c->plane = (long)c->rx * c->pitch;
  (void)hipGetDevice(&c->device);
  size_t pb = (size_t)c->plane * c->esize;
  bool ok = true;
  for (int i = 0; i < 2 && ok; i++) {
    ok = hipMalloc(&c->phi[i], pb * c->P) == hipSuccess && hipMalloc(&c->mu[i], pb * c->C) == hipSuccess &&
         (dtype == GP_F64 || hipMalloc(&c->mulo[i], pb * c->C) == hipSuccess);
    if (ok) ok = hipMemset(c->phi[i], 0, pb * c->P) == hipSuccess && hipMemset(c->mu[i], 0, pb * c->C) == hipSuccess &&
                 (dtype == GP_F64 || hipMemset(c->mulo[i], 0, pb * c->C) == hipSuccess);
  }
  ok = ok && hipMalloc(&c->dphi, pb * c->P) == hipSuccess && hipMemset(c->dphi, 0, pb * c->P) == hipSuccess;
  ok = ok && hipMalloc((void **)&c->dcode, (size_t)c->plane) == hipSuccess &&
       hipMemset(c->dcode, 0xff, (size_t)c->plane) == hipSuccess;
  {
    const dim3 gp = gpk::phase_grid(c->rx, c->ry);
    const size_t nsplit = 2 + (size_t)gp.x * gp.y + (size_t)((p->mesh_y + gpk::MW - 1) / gpk::MW) *
                                                        ((p->mesh_x + gpk::BY - 1) / gpk::BY);
    ok = ok && hipMalloc((void **)&c->dsplit, sizeof(int) * nsplit) == hipSuccess &&
         hipMemset(c->dsplit, 0, sizeof(int) * nsplit) == hipSuccess;
  }
  long ncell = p->mesh_x * p->mesh_y;
  c->nstat_blocks = (int)std::min<long>(1024, (ncell + 255) / 256);
  int nv = 3 * c->P + 3 * c->C + 1 + c->P + c->C + 4;  // k_stats accumulators (gp_run.hpp run_stats)
  ok = ok && hipMalloc((void **)&c->dpart, sizeof(double) * c->nstat_blocks * nv) == hipSuccess;
  if (ok && (p->mpi & GP_MPI_COMPOSITION))
    ok = hipMalloc(&c->dcomp, pb * c->C) == hipSuccess && hipMemset(c->dcomp, 0, pb * c->C) == hipSuccess;
  if (ok && (p->mpi & GP_MPI_NOISE) && p->noise) {
    const unsigned long long s0 = p->mpi_rand & gpk::kLcgMask;
    ok = hipMalloc((void **)&c->drstate, sizeof(unsigned long long)) == hipSuccess &&
         hipMemcpy(c->drstate, &s0, sizeof s0, hipMemcpyHostToDevice) == hipSuccess;
  }
  if (dtype == GP_F64) {
    gpk::DevParams<double> *h = new (std::nothrow) gpk::DevParams<double>();
    ok = ok && h;
    if (ok) {
      fill_devparams(*p, c->rx, c->ry, c->pitch, c->plane, *h);
      h->comp = (double *)c->dcomp;
      h->rstate = c->drstate;
      c->pow2 = h->pow2_dx && h->pow2_dy;
      ok = hipMalloc(&c->dprm, sizeof(*h)) == hipSuccess && hipMemcpy(c->dprm, h, sizeof(*h), hipMemcpyHostToDevice) == hipSuccess;
    }
    delete h;
  } else {
    gpk::DevParams<float> *h = new (std::nothrow) gpk::DevParams<float>();
    ok = ok && h;
    if (ok) {
      fill_devparams(*p, c->rx, c->ry, c->pitch, c->plane, *h);
      ok = hipMalloc(&c->dprm, sizeof(*h)) == hipSuccess && hipMemcpy(c->dprm, h, sizeof(*h), hipMemcpyHostToDevice) == hipSuccess;
    }
    delete h;
  }
  ok = ok && hipEventCreate(&c->ev0) == hipSuccess && hipEventCreate(&c->ev1) == hipSuccess;
  if (ok && p->noise && !p->mpi) {
    // one word per active phase of [1, rows-2]^2 at most
    c->nz_cap = (int)std::min<long>((long)c->P * (c->rx - 2) * (c->ry - 2), 0x7fffffffL);
    uint32_t st[31];
    noise_seed_state(1u, st);
    std::vector<uint32_t> jump;
    noise_jump_tables(jump);
    ok = hipMalloc((void **)&c->dnz_state, sizeof(uint32_t) * 31) == hipSuccess &&
         hipMalloc((void **)&c->dnz_jump, sizeof(uint32_t) * jump.size()) == hipSuccess &&
         // + one word per phase: a binary32 phase kernel whose activity test rounds
         // otherwise than the counting kernel's reads at most P words past the draws
         hipMalloc((void **)&c->dnz_raw, sizeof(uint32_t) * ((size_t)c->nz_cap + GP_MAX_PHASES)) == hipSuccess &&
         hipMalloc((void **)&c->dnz_off, sizeof(int) * (size_t)c->plane) == hipSuccess &&
         hipMalloc((void **)&c->dnz_rows, sizeof(int) * 2 * (size_t)c->rx) == hipSuccess &&
         hipMalloc((void **)&c->dnz_total, sizeof(int)) == hipSuccess &&
         hipMemcpy(c->dnz_state, st, sizeof st, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(c->dnz_jump, jump.data(), sizeof(uint32_t) * jump.size(), hipMemcpyHostToDevice) == hipSuccess;
  }
  // the fills and copies above run on the null stream, which the context's
  // non-blocking stream does not wait for: they finish before any of its work
  ok = ok && hipStreamSynchronize(nullptr) == hipSuccess;
  if (!ok) {
    free_ctx(c);
    return GP_E_NOMEM;
  }
  // a stream of our own (default priority) so that step blocks can be captured into graphs
  if (own_stream && hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking) != hipSuccess) {
    free_ctx(c);
    return GP_E_HIP;
  }
  c->stream = c->own_stream;
  c->cur = 0;
  c->path = 1;                            // automatic choice from the two-pass path on
  c->auto_mode = 1;
  c->use_graphs = p->isothermal ? 1 : 0;  // non-isothermal steps take per-step arguments (no graphs)
  c->graph_path = -1;
  c->shape = 0;
  c->shape_set = -1;
  for (int g = 0; g < GP_GRAPH_SLOTS; g++) c->gkey[g] = -1;
  c->auto_period = 64;
  if (p->mpi) c->auto_mode = 0;  // one kernel pair carries the MPI semantics
  *out = c;
  return GP_OK;
}

int gp_create(const gp_params *p, int dtype, gp_ctx **out) { return ctx_create(p, dtype, true, out); }

void gp_destroy(gp_ctx *c) {
  if (!c) return;
  (void)hipStreamSynchronize(c->stream);
  free_ctx(c);
}

int gp_set_stream(gp_ctx *c, void *s) {
  if (!c) return GP_E_ARG;
  c->stream = s ? (hipStream_t)s : c->own_stream;
  return GP_OK;
}

int gp_set_graphs(gp_ctx *c, int on) {
  if (!c) return GP_E_ARG;
  c->use_graphs = on != 0 && c->hp.isothermal;  // non-isothermal steps take per-step arguments
  return GP_OK;
}

int gp_set_path(gp_ctx *c, int path) {
  if (!c || path < -1 || path >= GP_NPATHS || (c->nmember && path != 3 && path != -1)) return GP_E_ARG;
  if (c->hp.mpi) {  // the MPI semantics run on their own two-pass kernels
    if (path != 1 && path != -1) return GP_E_UNSUPPORTED;
    c->path = 1;
    return GP_OK;
  }
  if ((!c->hp.isothermal || c->hp.noise) && path != 1 && path != 4 && path != 5 && path != 6 && path != -1)
    return GP_E_UNSUPPORTED;  // non-isothermal and noise runs step on the two-pass, split and one-hot paths
  c->auto_mode = path < 0;
  c->auto_count = 0;
  c->auto_next = 0;
  c->auto_gap = c->auto_period;
  c->path = path < 0 ? (c->nmember ? 3 : 1) : path;
  return GP_OK;
}

int gp_set_state(gp_ctx *c, const double *phi, const double *mu) {
  if (!c || !phi || !mu) return GP_E_ARG;
  size_t n = (size_t)c->hp.mesh_x * c->hp.mesh_y;
  Transit buf(c);
  double *d = buf.d;
  if (!d) return GP_E_NOMEM;
  int rc = GP_OK;
  if (hipMemcpyAsync(d, phi, sizeof(double) * n * c->P, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
      hipMemcpyAsync(d + n * c->P, mu, sizeof(double) * n * c->C, hipMemcpyHostToDevice, c->stream) != hipSuccess)
    rc = GP_E_HIP;
  if (!rc) rc = c->dtype == GP_F64 ? load_state<double, double>(c, d, d + n * c->P) : load_state<float, double>(c, d, d + n * c->P);
  if (!rc && c->dcomp) rc = comp_init(c);
  if (hipStreamSynchronize(c->stream) != hipSuccess && !rc) rc = GP_E_HIP;
  return rc;
}

int gp_get_state(gp_ctx *c, double *phi, double *mu) {
  if (!c || !phi || !mu) return GP_E_ARG;
  size_t n = (size_t)c->hp.mesh_x * c->hp.mesh_y;
  Transit buf(c);
  double *d = buf.d;
  if (!d) return GP_E_NOMEM;
  int rc = c->dtype == GP_F64 ? store_state<double, double>(c, d, d + n * c->P) : store_state<float, double>(c, d, d + n * c->P);
  if (!rc && (hipMemcpyAsync(phi, d, sizeof(double) * n * c->P, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
              hipMemcpyAsync(mu, d + n * c->P, sizeof(double) * n * c->C, hipMemcpyDeviceToHost, c->stream) != hipSuccess))
    rc = GP_E_HIP;
  if (hipStreamSynchronize(c->stream) != hipSuccess && !rc) rc = GP_E_HIP;
  return rc;
}

int gp_set_state_device(gp_ctx *c, const void *phi, const void *mu) {
  if (!c || !phi || !mu) return GP_E_ARG;
  int rc = c->dtype == GP_F64 ? load_state<double, double>(c, (const double *)phi, (const double *)mu)
                              : load_state<float, float>(c, (const float *)phi, (const float *)mu);
  if (!rc && c->dcomp) rc = comp_init(c);
  return rc;
}

int gp_set_composition(gp_ctx *c, const double *comp) {
  if (!c || !comp) return GP_E_ARG;
  if (!c->dcomp) return GP_E_UNSUPPORTED;
  for (int k = 0; k < c->C; k++) {
    const double *src = comp + (size_t)k * c->hp.mesh_x * c->hp.mesh_y;
    double *dst = (double *)c->dcomp + (size_t)k * c->plane + 3 * (size_t)c->pitch + 3;
    GP_HIP_CHECK(hipMemcpy2DAsync(dst, sizeof(double) * c->pitch, src, sizeof(double) * c->hp.mesh_y,
                                  sizeof(double) * c->hp.mesh_y, c->hp.mesh_x, hipMemcpyHostToDevice, c->stream));
  }
  // ghost images: the composition follows mu's copies
  GP_HIP_CHECK(comp_ghosts(c));
  GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  return GP_OK;
}

int gp_get_composition(gp_ctx *c, double *comp) {
  if (!c || !comp) return GP_E_ARG;
  if (!c->dcomp) return GP_E_UNSUPPORTED;
  for (int k = 0; k < c->C; k++) {
    double *dst = comp + (size_t)k * c->hp.mesh_x * c->hp.mesh_y;
    const double *src = (const double *)c->dcomp + (size_t)k * c->plane + 3 * (size_t)c->pitch + 3;
    GP_HIP_CHECK(hipMemcpy2DAsync(dst, sizeof(double) * c->hp.mesh_y, src, sizeof(double) * c->pitch,
                                  sizeof(double) * c->hp.mesh_y, c->hp.mesh_x, hipMemcpyDeviceToHost, c->stream));
  }
  GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  return GP_OK;
}

int gp_get_rand_state(gp_ctx *c, unsigned long long *state) {
  if (!c || !state) return GP_E_ARG;
  if (!c->drstate) return GP_E_UNSUPPORTED;
  GP_HIP_CHECK(hipMemcpyAsync(state, c->drstate, sizeof *state, hipMemcpyDeviceToHost, c->stream));
  GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  return GP_OK;
}

int gp_get_state_device(gp_ctx *c, void *phi, void *mu) {
  if (!c || !phi || !mu) return GP_E_ARG;
  return c->dtype == GP_F64 ? store_state<double, double>(c, (double *)phi, (double *)mu)
                            : store_state<float, float>(c, (float *)phi, (float *)mu);
}

// Binary64 steps: the power-of-two build (namespace gpk2) for P <= 4, where it
// was measured faster (C2: -8% on the split path, -19% on the two-pass path);
// at P = 9 its phase kernel spills more and the general build is faster.
#define GP_POW2_MAX_P 4
}  // extern "C"
template <int P, int C>
static int steps_f64(gp_ctx *c, long nsteps) {
  if constexpr (P <= GP_POW2_MAX_P) {
    if (c->pow2) return gpk2::run_steps<P, C, double>(c, nsteps);
  }
  return gpk::run_steps<P, C, double>(c, nsteps);
}
extern "C" {

static int dispatch_steps(gp_ctx *c, long nsteps) {
  int rc = GP_E_UNSUPPORTED;
  if (c->path >= 0 && c->path < GP_NPATHS) c->path_steps[c->path] += nsteps;
#define GP_DISPATCH_STEP(P_, C_)                                                                   \
  if (c->P == P_ && c->C == C_)                                                                    \
    rc = c->dtype == GP_F32 ? gpk::run_steps<P_, C_, float>(c, nsteps) : steps_f64<P_, C_>(c, nsteps);
  GP_PC_LIST(GP_DISPATCH_STEP)
#undef GP_DISPATCH_STEP
  return rc;
}

// Graph cache slot of the current (path, tile shape).
static int graph_slot(gp_ctx *c) {
  const int key = c->path * 16 + c->shape;
  for (int g = 0; g < GP_GRAPH_SLOTS; g++)
    if (c->gkey[g] == key) return g;
  for (int g = 0; g < GP_GRAPH_SLOTS; g++)
    if (c->gkey[g] < 0) {
      c->gkey[g] = key;
      return g;
    }
  // evict slot 0; a replay of it may still be queued
  (void)hipStreamSynchronize(c->stream);
  for (int i = 0; i < 2; i++)
    if (c->gcache[0][i]) (void)hipGraphExecDestroy(c->gcache[0][i]), c->gcache[0][i] = nullptr;
  c->gkey[0] = key;
  return 0;
}

// Capture GP_GRAPH_STEPS steps starting from the current buffer parity.  The
// block length is even, so after it the parities (state buffers, tile flags,
// counters) are back where they started and the graph can be replayed.
static int capture_graph(gp_ctx *c, int gi) {
  const int slot = c->cur;
  if (c->gcache[gi][slot]) return GP_OK;
  int cur0 = c->cur, par0 = c->cnt_par, fv0 = c->flags_valid, ov0 = c->oh_valid;
  const long counted0 = c->path_steps[c->path];  // captured steps are not run steps
  hipGraph_t g;
  GP_HIP_CHECK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  int rc = dispatch_steps(c, GP_GRAPH_STEPS);
  hipError_t e = hipStreamEndCapture(c->stream, &g);
  c->cur = cur0;
  c->cnt_par = par0;
  c->flags_valid = fv0;
  c->oh_valid = ov0;
  c->path_steps[c->path] = counted0;
  if (rc) return rc;
  if (e != hipSuccess) return GP_E_HIP;
  e = hipGraphInstantiate(&c->gcache[gi][slot], g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  return e == hipSuccess ? GP_OK : GP_E_HIP;
}

// One block of GP_GRAPH_STEPS steps with the current path as a graph replay.
static int run_block(gp_ctx *c) {
  int rc = dispatch_steps(c, 0);  // tile set and flags of the current state, outside the capture
  if (rc) return rc;
  const int gi = graph_slot(c);
  if ((rc = capture_graph(c, gi))) return rc;
  if (hipGraphLaunch(c->gcache[gi][c->cur], c->stream) != hipSuccess) return GP_E_HIP;
  c->path_steps[c->path] += GP_GRAPH_STEPS;
  if (c->path == 1 || c->path >= 4) c->flags_valid = 0;  // the two-pass kernels keep no tile flags
  return GP_OK;
}

// Automatic path choice: one timed block of each candidate (real steps of the
// run), then the fastest is kept until the next re-timing.  The candidates are
// the two-pass, split, compact split and one-hot paths; the sparse tile paths
// (0, 3), slower than these on every single-grid workload measured, are left
// to explicit choice, since a timed block of a slow path costs its real steps.
static int retune(gp_ctx *c, long *left) {
  const int cand[4] = {1, 4, 5, 6};
  const int ncand = c->nmember ? 1 : 4;
  double best = 1e300;
  int pick = c->path;
  hipEvent_t a = c->ev0, b = c->ev1;
  hipEvent_t t0, t1;
  if (hipEventCreate(&t0) != hipSuccess) return GP_E_HIP;
  if (hipEventCreate(&t1) != hipSuccess) {
    (void)hipEventDestroy(t0);
    return GP_E_HIP;
  }
  (void)a;
  (void)b;
  int rc = GP_OK;
  for (int i = 0; i < ncand && *left >= GP_GRAPH_STEPS; i++) {
    c->path = c->nmember ? 3 : cand[i];
    c->shape = 0;
    if ((rc = dispatch_steps(c, 0))) break;
    const int gi = graph_slot(c);
    if ((rc = capture_graph(c, gi))) break;
    if (hipEventRecord(t0, c->stream) != hipSuccess || hipGraphLaunch(c->gcache[gi][c->cur], c->stream) != hipSuccess ||
        hipEventRecord(t1, c->stream) != hipSuccess || hipEventSynchronize(t1) != hipSuccess) {
      rc = GP_E_HIP;
      break;
    }
    c->path_steps[c->path] += GP_GRAPH_STEPS;
    if (c->path == 1 || c->path >= 4) c->flags_valid = 0;
    float ms = 0;
    (void)hipEventElapsedTime(&ms, t0, t1);
    if (ms < best) {
      best = ms;
      pick = c->path;
    }
    *left -= GP_GRAPH_STEPS;
  }
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  c->path = pick;
  return rc;
}

// Automatic choice without graphs (graphs off, the default stream, or a
// non-isothermal context): one timed 32-step block of eager launches of each
// candidate, real steps of the run.  Counts the steps it takes in tstep.
static int retune_eager(gp_ctx *c, long *left) {
  const int cand[4] = {1, 4, 5, 6};  // as in retune
  const int ncand = c->nmember ? 1 : 4;
  double best = 1e300;
  int pick = c->path;
  hipEvent_t t0, t1;
  if (hipEventCreate(&t0) != hipSuccess) return GP_E_HIP;
  if (hipEventCreate(&t1) != hipSuccess) {
    (void)hipEventDestroy(t0);
    return GP_E_HIP;
  }
  int rc = GP_OK;
  for (int i = 0; i < ncand && *left >= GP_GRAPH_STEPS; i++) {
    c->path = c->nmember ? 3 : cand[i];
    c->shape = 0;
    if (hipEventRecord(t0, c->stream) != hipSuccess) { rc = GP_E_HIP; break; }
    if ((rc = dispatch_steps(c, GP_GRAPH_STEPS))) break;
    if (hipEventRecord(t1, c->stream) != hipSuccess || hipEventSynchronize(t1) != hipSuccess) { rc = GP_E_HIP; break; }
    c->tstep += GP_GRAPH_STEPS;
    c->shift_pend = 0;
    float ms = 0;
    (void)hipEventElapsedTime(&ms, t0, t1);
    if (ms < best) {
      best = ms;
      pick = c->path;
    }
    *left -= GP_GRAPH_STEPS;
  }
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  c->path = pick;
  return rc;
}

int gp_step(gp_ctx *c, long nsteps) { return gp_step_impl(c, nsteps, true); }

}  // extern "C"

// Steps without the closing synchronisation when `timed` is false (callers that
// queue more work, such as the adjoint's recomputation).
int gp_step_impl(gp_ctx *c, long nsteps, bool timed) {
  if (!c || nsteps < 0) return GP_E_ARG;
  if (timed) GP_HIP_CHECK(hipEventRecord(c->ev0, c->stream));
  int rc = GP_OK;
  long left = nsteps;
  // graphs: on a capturable stream, for runs of at least one block
  if (c->use_graphs && c->stream && left >= GP_GRAPH_STEPS) {
    while (!rc && left >= GP_GRAPH_STEPS) {
      if (c->auto_mode && c->auto_count >= c->auto_next && left >= 3 * GP_GRAPH_STEPS) {
        const int before = c->path;
        const bool first = c->auto_count == 0;
        rc = retune(c, &left);
        c->auto_count++;
        c->auto_gap = (!first && c->path == before) ? std::min(2 * c->auto_gap, 8 * c->auto_period) : c->auto_period;
        c->auto_next = c->auto_count + c->auto_gap;
        continue;
      }
      c->auto_count++;
      rc = run_block(c);
      left -= GP_GRAPH_STEPS;
    }
  }
  long counted = 0;  // steps already added to tstep (the eager automatic choice)
  if (!rc && c->auto_mode && !(c->use_graphs && c->stream)) {
    while (!rc && left >= GP_GRAPH_STEPS) {
      if (c->auto_count >= c->auto_next && left >= 3 * GP_GRAPH_STEPS) {
        const int before = c->path;
        const bool first = c->auto_count == 0;
        const long l0 = left;
        rc = retune_eager(c, &left);
        counted += l0 - left;
        c->auto_count++;
        c->auto_gap = (!first && c->path == before) ? std::min(2 * c->auto_gap, 8 * c->auto_period) : c->auto_period;
        c->auto_next = c->auto_count + c->auto_gap;
        continue;
      }
      // up to the next re-timing in one dispatch
      const long blocks = std::max(1L, std::min(left / GP_GRAPH_STEPS, c->auto_next - c->auto_count));
      const long n = blocks * GP_GRAPH_STEPS;
      rc = dispatch_steps(c, n);
      c->tstep += n;
      c->shift_pend = 0;
      counted += n;
      left -= n;
      c->auto_count += blocks;
    }
  }
  if (!rc && left > 0) rc = dispatch_steps(c, left);
  if (rc) return rc;
  if (nsteps > 0) c->stepped = 1;
  c->tstep += nsteps - counted;
  if (nsteps > 0) c->shift_pend = 0;
  for (int i = 0; i < c->nmember; i++) {
    c->member[i]->cur = c->cur;
    c->member[i]->stepped = c->stepped;
  }
  if (!timed) return GP_OK;
  GP_HIP_CHECK(hipEventRecord(c->ev1, c->stream));
  GP_HIP_CHECK(hipEventSynchronize(c->ev1));
  float ms = 0;
  GP_HIP_CHECK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->last_ms = ms;
  return GP_OK;
}

// ------------------------------------------------- steps without allocation

// Cell lists of gp_step_noalloc: one array per device, held until the process
// ends.  Host code never passes `scratch` itself to a kernel (in host code the
// name is a stand-in, not a device address): each device's address comes from
// hipGetSymbolAddress with that device current, once, and is kept in
// scratch_dev.
#define GP_NOALLOC_SCRATCH_BYTES (64u << 20)
static __device__ __align__(256) int scratch[GP_NOALLOC_SCRATCH_BYTES / sizeof(int)];

static constexpr int kScratchDevices = 64;
static std::mutex scratch_mu;
static int *scratch_dev[kScratchDevices];

// Address of the current device's scratch array.
static int scratch_ptr(int dev, int **out) {
  if (dev < 0 || dev >= kScratchDevices) return GP_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_dev[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return GP_E_HIP;
    scratch_dev[dev] = (int *)p;
  }
  *out = scratch_dev[dev];
  return GP_OK;
}

template <int P, int C>
static int lists_f64(gp_ctx *c, long nsteps, int *cells) {
  if constexpr (P <= GP_POW2_MAX_P) {
    if (c->pow2) return gpk2::run_steps_lists<P, C, double>(c, nsteps, cells);
  }
  return gpk::run_steps_lists<P, C, double>(c, nsteps, cells);
}

extern "C" {

int gp_step_noalloc(gp_ctx *c, long nsteps) {
  if (!c || nsteps < 0 || c->nmember) return GP_E_ARG;
  const size_t ints = 2 + (size_t)(c->rx - 4) * (c->ry - 4) + (size_t)c->hp.mesh_x * c->hp.mesh_y;
  if (ints * sizeof(int) > GP_NOALLOC_SCRATCH_BYTES) return GP_E_SCRATCH;
  int dev = -1;
  GP_HIP_CHECK(hipGetDevice(&dev));
  const bool other = dev != c->device;
  if (other) GP_HIP_CHECK(hipSetDevice(c->device));
  int *cells = nullptr;
  int rc = scratch_ptr(c->device, &cells);
  if (!rc) {
    rc = GP_E_UNSUPPORTED;
#define GP_DISPATCH_LISTS(P_, C_)                                                                  \
  if (c->P == P_ && c->C == C_)                                                                    \
    rc = c->dtype == GP_F32 ? gpk::run_steps_lists<P_, C_, float>(c, nsteps, cells) : lists_f64<P_, C_>(c, nsteps, cells);
    GP_PC_LIST(GP_DISPATCH_LISTS)
#undef GP_DISPATCH_LISTS
  }
  if (!rc && nsteps > 0) {
    c->stepped = 1;
    c->tstep += nsteps;
    c->shift_pend = 0;
  }
  if (other) (void)hipSetDevice(dev);
  return rc;
}

int gp_path_steps(gp_ctx *c, long *steps, int reset) {
  if (!c) return GP_E_ARG;
  for (int i = 0; i < GP_NPATHS; i++) {
    if (steps) steps[i] = c->path_steps[i];
    if (reset) c->path_steps[i] = 0;
  }
  return GP_OK;
}

int gp_get_path(gp_ctx *c, int *path, int *automatic) {
  if (!c) return GP_E_ARG;
  if (path) *path = c->path;
  if (automatic) *automatic = c->auto_mode;
  return GP_OK;
}

int gp_set_tile_shape(gp_ctx *c, int shape) {
  if (!c || shape < 0 || shape >= gpk::kNumShapes) return GP_E_ARG;
  if (shape != 0 && c->P > 4) return GP_E_UNSUPPORTED;
  c->shape = shape;
  return GP_OK;
}

int gp_tile_shape(gp_ctx *c, int *tile_x, int *tile_y) {
  if (!c) return GP_E_ARG;
  int rc = dispatch_steps(c, 0);  // builds the tile set of the current path and shape
  if (rc) return rc;
  if (tile_x) *tile_x = c->tile_tx;
  if (tile_y) *tile_y = c->tile_ty;
  return GP_OK;
}

// Time `steps` steps of every candidate (path, tile shape) and keep the
// fastest.  The state advances by two runs of `steps` steps per candidate; all
// candidates give bit-identical binary64 results.
static int autotune(gp_ctx *c, long steps, bool paths) {
  struct Cand { int path, shape; };
  Cand cand[gpk::kNumShapes + 5];
  int n = 0;
  for (int s = 0; s < gpk::kNumShapes; s++)
    if (s == 0 || c->P <= 4) cand[n++] = {3, s};
  if (paths) {
    cand[n++] = {0, 0};
    cand[n++] = {1, 0};
    cand[n++] = {4, 0};
    cand[n++] = {5, 0};
    cand[n++] = {6, 0};
  }
  double best = 1e300;
  c->auto_mode = 0;
  Cand pick = {c->path, c->shape};
  for (int i = 0; i < n; i++) {
    c->path = cand[i].path;
    c->shape = cand[i].shape;
    int rc = gp_step(c, steps);  // warm-up: tile set, graph capture
    if (!rc) rc = gp_step(c, steps);
    if (rc) return rc;
    if (c->last_ms < best) {
      best = c->last_ms;
      pick = cand[i];
    }
  }
  c->path = pick.path;
  c->shape = pick.shape;
  return GP_OK;
}

int gp_autotune(gp_ctx *c, long steps, int *path, int *shape) {
  if (!c || steps < 1 || c->nmember) return GP_E_ARG;
  if (!c->hp.isothermal || c->hp.noise) return GP_E_UNSUPPORTED;
  int rc = autotune(c, steps, true);
  if (rc) return rc;
  if (path) *path = c->path;
  if (shape) *shape = c->shape;
  return GP_OK;
}

int gp_smooth(gp_ctx *c, long nsweeps) {
  if (!c || nsweeps < 0 || c->nmember) return GP_E_ARG;
  if (!c->hp.isothermal && nsweeps > 0) return GP_E_UNSUPPORTED;
  if (c->hp.mpi && nsweeps > 0) return GP_E_UNSUPPORTED;  // the MPI solver smooths in one fused sweep
  int rc = GP_E_UNSUPPORTED;
#define GP_DISPATCH_SMOOTH(P_, C_)                                                                  \
  if (c->P == P_ && c->C == C_)                                                                     \
    rc = c->dtype == GP_F64 ? gpk::run_smooth<P_, C_, double>(c, nsweeps) : gpk::run_smooth<P_, C_, float>(c, nsweeps);
  GP_PC_LIST(GP_DISPATCH_SMOOTH)
#undef GP_DISPATCH_SMOOTH
  if (!rc && nsweeps > 0) c->stepped = 1;
  if (!rc) GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  return rc;
}

int gp_sched_info(gp_ctx *c, long *ntiles, long *n_if, long *n_bulk) {
  if (!c) return GP_E_ARG;
  int cnt[2] = {0, 0};
  if (c->dcnt) {
    GP_HIP_CHECK(hipStreamSynchronize(c->stream));
    // counters of the last step: parity before the last flip
    GP_HIP_CHECK(hipMemcpy(cnt, c->dcnt + 2 * (c->cnt_par ^ 1), sizeof(cnt), hipMemcpyDeviceToHost));
  }
  if (ntiles) *ntiles = c->ntiles;
  if (n_if) *n_if = c->path == 2 ? c->ntiles : cnt[0];
  if (n_bulk) *n_bulk = c->path == 2 ? 0 : cnt[1];
  return GP_OK;
}

int gp_last_step_ms(gp_ctx *c, double *ms) {
  if (!c || !ms) return GP_E_ARG;
  *ms = c->last_ms;
  return GP_OK;
}

int gp_synchronize(gp_ctx *c) {
  if (!c) return GP_E_ARG;
  return hipStreamSynchronize(c->stream) == hipSuccess ? GP_OK : GP_E_HIP;
}

int gp_stats_get(gp_ctx *c, gp_stats *st) {
  if (!c || !st) return GP_E_ARG;
  memset(st, 0, sizeof(*st));
  int rc = GP_E_UNSUPPORTED;
#define GP_DISPATCH_STATS(P_, C_)                                                                 \
  if (c->P == P_ && c->C == C_)                                                                   \
    rc = c->dtype == GP_F64 ? gpk::run_stats<P_, C_, double>(c, st) : gpk::run_stats<P_, C_, float>(c, st);
  GP_PC_LIST(GP_DISPATCH_STATS)
#undef GP_DISPATCH_STATS
  if (rc) return rc;
  return st->nonfinite > 0 ? GP_E_NONFINITE : GP_OK;
}

// -------------------------------------------------------------- moving frame

}  // extern "C"

template <class R>
static int frame_pos(gp_ctx *c, long *pos) {
  const gpk::DevParams<R> *prm = (const gpk::DevParams<R> *)c->dprm;
  const long MX = c->hp.mesh_x;
  if (!c->drow && hipMalloc((void **)&c->drow, sizeof(int) * MX) != hipSuccess) {
    c->drow = nullptr;
    return GP_E_NOMEM;
  }
  hipLaunchKernelGGL((gpk::k_iface_rows<R>), dim3((unsigned)MX), dim3(gpk::IFB), 0, c->stream, prm,
                     (const R *)c->phi[c->cur] + (size_t)(c->P - 1) * c->plane, c->drow);
  GP_HIP_CHECK(hipGetLastError());
  std::vector<int> h((size_t)MX);
  GP_HIP_CHECK(hipMemcpyAsync(h.data(), c->drow, sizeof(int) * MX, hipMemcpyDeviceToHost, c->stream));
  GP_HIP_CHECK(hipStreamSynchronize(c->stream));
  int m = 0;
  for (int v : h) m = std::max(m, v);
  *pos = m;
  return GP_OK;
}

template <class R>
static int frame_shift(gp_ctx *c, int d, const double *mu_fill) {
  const gpk::DevParams<R> *prm = (const gpk::DevParams<R> *)c->dprm;
  const dim3 blk(gpk::BX, gpk::BY), g((c->ry + gpk::BX - 1) / gpk::BX, (c->rx + gpk::BY - 1) / gpk::BY);
  gpk::ShiftFill fp = {}, fm = {}, fz = {};
  fp.v[c->P - 1] = 1.0;
  for (int k = 0; k < c->C; k++) fm.v[k] = mu_fill[k];
  const int o = c->cur ^ 1;
  hipLaunchKernelGGL((gpk::k_shift_y<R>), g, blk, 0, c->stream, prm, (const R *)c->phi[c->cur], (R *)c->phi[o], c->P, d, fp);
  hipLaunchKernelGGL((gpk::k_shift_y<R>), g, blk, 0, c->stream, prm, (const R *)c->mu[c->cur], (R *)c->mu[o], c->C, d, fm);
  if (c->mulo[c->cur])
    hipLaunchKernelGGL((gpk::k_shift_y<R>), g, blk, 0, c->stream, prm, (const R *)c->mulo[c->cur], (R *)c->mulo[o], c->C, d, fz);
  GP_HIP_CHECK(hipGetLastError());
  c->cur = o;
  return GP_OK;
}

extern "C" {

int gp_check_shift(gp_ctx *c, long *pos) {
  if (!c || !pos || c->nmember > 0 || !c->phi[0]) return GP_E_ARG;
  return c->dtype == GP_F64 ? frame_pos<double>(c, pos) : frame_pos<float>(c, pos);
}

int gp_apply_shift_y(gp_ctx *c, long d, const double *mu_fill) {
  if (!c || !mu_fill || c->nmember > 0 || !c->phi[0]) return GP_E_ARG;
  if (d < 1 || d > c->hp.mesh_y) return GP_E_ARG;
  for (int k = 0; k < c->C; k++)
    if (!isfinite(mu_fill[k])) return GP_E_ARG;
  int rc = c->dtype == GP_F64 ? frame_shift<double>(c, (int)d, mu_fill) : frame_shift<float>(c, (int)d, mu_fill);
  if (rc) return rc;
  c->shift_off += d;
  c->shift_pend += d;
  c->stepped = 0;
  c->flags_valid = 0;
  c->oh_valid = 0;
  return GP_OK;
}

// ------------------------------------------------------------------ ensembles

struct gp_ensemble {
  gp_ctx *m;  // master: the tile set over all members, stream, events, graphs
};

static void free_ensemble(gp_ensemble *e) {
  if (!e) return;
  if (e->m) {
    // the master's captured blocks name the members' buffers: they go first
    if (e->m->stream) (void)hipStreamSynchronize(e->m->stream);
    release_graphs(e->m);
    for (int i = 0; i < e->m->nmember; i++)
      if (e->m->member[i]) free_ctx(e->m->member[i]);
    delete[] e->m->member;
    e->m->nmember = 0;
    free_ctx(e->m);
  }
  delete e;
}

int gp_ensemble_create(const gp_params *params, int n, int dtype, gp_ensemble **out) {
  if (!params || !out || n < 1 || (dtype != GP_F64 && dtype != GP_F32)) return GP_E_ARG;
  *out = nullptr;
  for (int i = 1; i < n; i++)
    if (params[i].nphases != params[0].nphases || params[i].ncomp != params[0].ncomp) return GP_E_ARG;
  if (!pc_supported(params[0].nphases, params[0].ncomp)) return GP_E_UNSUPPORTED;
  for (int i = 0; i < n; i++)
    if (!params[i].isothermal || params[i].noise) return GP_E_UNSUPPORTED;
  gp_ensemble *e = new (std::nothrow) gp_ensemble();
  if (!e) return GP_E_NOMEM;
  gp_ctx *m = e->m = new (std::nothrow) gp_ctx();
  if (!m) {
    delete e;
    return GP_E_NOMEM;
  }
  m->member = new (std::nothrow) gp_ctx *[n]();
  if (!m->member) {
    free_ensemble(e);
    return GP_E_NOMEM;
  }
  m->nmember = n;
  m->hp = params[0];
  m->dtype = dtype;
  m->P = params[0].nphases;
  m->C = params[0].ncomp;
  m->esize = dtype == GP_F64 ? 8 : 4;
  (void)hipGetDevice(&m->device);
  if (hipStreamCreateWithFlags(&m->own_stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess) {
    free_ensemble(e);
    return GP_E_HIP;
  }
  m->stream = m->own_stream;
  m->path = 3;
  m->use_graphs = 1;
  m->graph_path = -1;
  m->shape = 0;
  m->shape_set = -1;
  for (int g = 0; g < GP_GRAPH_SLOTS; g++) m->gkey[g] = -1;
  m->auto_period = 64;
  for (int i = 0; i < n; i++) {
    int rc = ctx_create(&params[i], dtype, false, &m->member[i]);
    if (rc) {
      free_ensemble(e);
      return rc;
    }
    m->member[i]->stream = m->stream;
    m->member[i]->stage_of = m;
    m->stage_bytes = std::max(m->stage_bytes, m->member[i]->stage_bytes);
  }
  // the power-of-two build steps an ensemble whose members all allow it
  m->pow2 = 1;
  for (int i = 0; i < n; i++) m->pow2 = m->pow2 && m->member[i]->pow2;
  *out = e;
  return GP_OK;
}

void gp_ensemble_destroy(gp_ensemble *e) {
  if (!e) return;
  if (e->m) (void)hipStreamSynchronize(e->m->stream);
  free_ensemble(e);
}

int gp_ensemble_size(gp_ensemble *e, int *n, long *cells) {
  if (!e) return GP_E_ARG;
  long s = 0;
  for (int i = 0; i < e->m->nmember; i++) s += e->m->member[i]->hp.mesh_x * e->m->member[i]->hp.mesh_y;
  if (n) *n = e->m->nmember;
  if (cells) *cells = s;
  return GP_OK;
}

int gp_ensemble_set_state(gp_ensemble *e, int i, const double *phi, const double *mu) {
  if (!e || i < 0 || i >= e->m->nmember) return GP_E_ARG;
  gp_ctx *g = e->m->member[i];
  g->cur = e->m->cur;
  int rc = gp_set_state(g, phi, mu);
  e->m->flags_valid = 0;
  e->m->stepped = 0;
  for (int k = 0; k < e->m->nmember; k++) e->m->member[k]->stepped = 0;
  return rc;
}

int gp_ensemble_get_state(gp_ensemble *e, int i, double *phi, double *mu) {
  if (!e || i < 0 || i >= e->m->nmember) return GP_E_ARG;
  return gp_get_state(e->m->member[i], phi, mu);
}

int gp_ensemble_step(gp_ensemble *e, long nsteps) {
  if (!e) return GP_E_ARG;
  return gp_step(e->m, nsteps);
}

int gp_ensemble_stats_get(gp_ensemble *e, int i, gp_stats *st) {
  if (!e || i < 0 || i >= e->m->nmember) return GP_E_ARG;
  return gp_stats_get(e->m->member[i], st);
}

int gp_ensemble_last_step_ms(gp_ensemble *e, double *ms) {
  if (!e || !ms) return GP_E_ARG;
  *ms = e->m->last_ms;
  return GP_OK;
}

int gp_ensemble_set_tile_shape(gp_ensemble *e, int shape) {
  if (!e) return GP_E_ARG;
  return gp_set_tile_shape(e->m, shape);
}

int gp_ensemble_autotune(gp_ensemble *e, long steps, int *tile_x, int *tile_y) {
  if (!e || steps < 1) return GP_E_ARG;
  int rc = autotune(e->m, steps, false);
  if (!rc) rc = gp_tile_shape(e->m, tile_x, tile_y);
  return rc;
}

int gp_ensemble_sched_info(gp_ensemble *e, long *ntiles, long *n_interface, long *n_bulk, int *tile_x, int *tile_y) {
  if (!e) return GP_E_ARG;
  int rc = gp_tile_shape(e->m, tile_x, tile_y);
  if (!rc) rc = gp_sched_info(e->m, ntiles, n_interface, n_bulk);
  return rc;
}

int gp_ensemble_synchronize(gp_ensemble *e) {
  if (!e) return GP_E_ARG;
  return gp_synchronize(e->m);
}

// sizes of the ABI structures, so bindings can check their layouts
int gp_abi_sizes(size_t *params, size_t *stats, size_t *input) {
  if (params) *params = sizeof(gp_params);
  if (stats) *stats = sizeof(gp_stats);
  if (input) *input = sizeof(gp_input);
  return GP_OK;
}

}  // extern "C"
