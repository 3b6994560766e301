// Element assembly (matrix_fill_full) for QUAD9 / HEX27 Q2-P1 Navier-Stokes
// with optional energy, as HIP kernels for gfx950.
//
// k_elem2 (QUAD9, four elements per workgroup) and k_elem3 (HEX27, one) form
// the element matrices and vectors; k_gather (gm_gather.hip) sums them into
// the rows: deterministic, no atomics.
//
// Per element:
//   1. nodal coordinates / unknowns -> LDS
//   2. per quadrature point: map Jacobian, inverse, dA = detJ*w  (beer_belly)
//   3. physical basis gradients grad_phi[q][k][p]                (load_bf_grad)
//   4. per quadrature point: v, grad v, T, grad T, P, mu(gammadot), body force
//   5. residual rows, then the Jacobian: the node-by-node blocks as products
//      over the quadrature points on the FP64 matrix cores, pressure couplings
//      as separate tasks.
//   6. Dirichlet rows: J row -> unit diagonal, R -> x - V (per element, as
//      put_dirichlet_in_matrix does, src/bc_dirich.c:44-153), in the scatter.
//   7. scatter into the MSR arrays.
//
// Weak forms (Goma's, restated):
//   momentum  (src/mm_fill_momentum.c:474-672, J_m_v 1564-1735, J_m_T 746-915,
//             J_m_P 2052-2117; fluid_stress 2834-3737):
//     R_a,i = int[ -rho phi_i (v.grad v_a) - grad phi_i . Pi[a][.] + phi_i f_a ] dA
//     Pi = -P I + mu (grad v + grad v^T),  f_a = -rho g_a beta (T - Tref)
//   continuity (src/mm_fill_continuity.c:435-700):  R_k = int psi_k div v dA
//     with PSPG (global tau, src/mm_fill_continuity.c:600-612; calc_pspg
//     src/mm_fill_stabilization.c:1037-1049, 1100-1465, no polymer stress):
//     R_k += int grad psi_k . tau (rho v_dot + rho v.grad v + grad P - f) dA,
//     grad psi_0 = 0 and grad psi_k = B[.][k-1] for the P1 basis {1, xi_k}
//   energy   (src/mm_fill_energy.c:280-700, heat_flux 1629):
//     R_i = int[ -rho Cp w_i (v.grad T) - k grad phi_i . grad T + phi_i h ] dA
//     w_i = phi_i, or with SUPG (src/mm_fill_energy.c:237-259, 332-339)
//     w_i = phi_i + s/h (v.grad phi_i), h = sqrt(sum_p vc_p^2 / hsq_p) / 2
//     from the squared face-centroid widths hsq and the velocity vc at the
//     element's last local node (element_velocity, src/mm_fill_aux.c:798)
#include <cmath>
#include <vector>

#include "gm_launch.h"

template <int DIM>
struct El {
  static constexpr int NVE = DIM == 2 ? 9 : 27;
  static constexpr int NQ = DIM == 2 ? 9 : 27;
  static constexpr int NP = DIM + 1;
};

struct FillArgs {
  const double *coor;       // [dim][num_nodes]
  const int *conn;          // [num_elems][nve]
  const int *fu;            // first unknown per node
  const int *centroid;      // centroid node per element
  const double *tables;     // phi, dphidxi, psi, wt
  const double *x;
  double *re, *ct;  // element residuals, PSPG continuity x temperature entries
  // [num_elems][E]: element matrices before the Dirichlet rows (also for the
  // Galerkin multigrid coarse operators): nodal blocks [a][i][j][b] (variable b
  // innermost: a node pair's row a is one access of the kernels that read it),
  // then momentum x P, continuity x velocity, P x P as in the e2nz map
  double *kel;
  int *flag;
  // theta-method time step (nullptr x_old: steady): at each node
  // xdot = cmass (x - x_old) - cold xdot_old, cmass = (1 + 2 theta) / dt, cold = 2 theta
  const double *x_old, *xdot_old;
  double cmass, cold;
  // QSIDE / QCONV side entries: those of element e are [qs_ptr[e], qs_ptr[e+1]),
  // each a side number (1-based, Exodus order) and (q, h, T_c) at qs_q[3 k]:
  // inward heat flux q + h (T_c - T); nullptr qs_ptr: none
  const int *qs_ptr, *qs_side;
  const double *qs_q;
  const double *stab;  // side tables: [side][point] phi[NVE], dphidxi[NVE][DIM], weight
  int num_nodes;
  double tau_pspg;  // global PSPG tau, 0: no pressure stabilisation
  double supg_e;    // energy SUPG coefficient, 0: Galerkin weights
  int resid_only;  // 1: residual only (Assemble_Jacobian = FALSE)
  long long E;
  long long off_mp, off_cv, off_cp;
  double rho, mu0, muinf, lam, nexp, aexp, Cp, kcond, hsrc, g[3], beta, Tref;
};

// Reference tables: phi[NQ][NVE], dphidxi[NQ][NVE][DIM], psi[NQ][NP], wt[NQ].
template <int DIM>
struct Tab {
  static constexpr int NVE = El<DIM>::NVE, NQ = El<DIM>::NQ, NP = El<DIM>::NP;
  static constexpr int PHI = 0;
  static constexpr int DPHI = PHI + NQ * NVE;
  static constexpr int PSI = DPHI + NQ * NVE * DIM;
  static constexpr int WT = PSI + NQ * NP;
  static constexpr int SIZE = WT + NQ;
};

// Side tables for surface integrals (QSIDE): for each of the 2*DIM sides in
// Exodus order and each surface Gauss point (3-point rule per free axis),
// phi[NVE], dphidxi[NVE][DIM] and the weight.
template <int DIM>
struct STab {
  static constexpr int NVE = El<DIM>::NVE;
  static constexpr int NSIDE = 2 * DIM;
  static constexpr int NSP = DIM == 2 ? 3 : 9;
  static constexpr int REC = NVE + NVE * DIM + 1;
  static constexpr int SIZE = NSIDE * NSP * REC;
};

// Energy SUPG element parameters (src/mm_fill_energy.c:250-259, 644-651):
// out[0] = s / h, out[1 + b] = s d(1/h)/d vc_b (the derivative in the
// velocity component b at the last local node), all zero when h = 0.  x are
// the element's nodal coordinates (local order), vc the velocity at the last
// local node.  Face-centroid widths as h_elem_siz (src/mm_fill_aux.c:844).
template <int DIM, typename XA>
__device__ inline void supg_params(double s, const XA &x, const double *vc, double *out) {
  double hsq[3];
  if constexpr (DIM == 2) {
    double w0 = 0.0, w1 = 0.0;
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const double d0 = 0.5 * (x[a][1] + x[a][2]) - 0.5 * (x[a][0] + x[a][3]);
      const double d1 = 0.5 * (x[a][0] + x[a][1]) - 0.5 * (x[a][2] + x[a][3]);
      w0 += d0 * d0;
      w1 += d1 * d1;
    }
    hsq[0] = w0;
    hsq[1] = w1;
  } else {
    double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const double f1 = 0.25 * (x[a][0] + x[a][1] + x[a][2] + x[a][3]);
      const double f2 = 0.25 * (x[a][1] + x[a][2] + x[a][5] + x[a][6]);
      const double f3 = 0.25 * (x[a][2] + x[a][3] + x[a][6] + x[a][7]);
      const double f4 = 0.25 * (x[a][0] + x[a][1] + x[a][4] + x[a][5]);
      const double f5 = 0.25 * (x[a][0] + x[a][3] + x[a][4] + x[a][7]);
      const double f6 = 0.25 * (x[a][4] + x[a][5] + x[a][6] + x[a][7]);
      w[0] += (f2 - f5) * (f2 - f5);
      w[1] += (f3 - f4) * (f3 - f4);
      w[2] += (f1 - f6) * (f1 - f6);
    }
    hsq[0] = w[0];
    hsq[1] = w[1];
    hsq[2] = w[2];
  }
  double he = 0.0;
#pragma unroll
  for (int p = 0; p < DIM; p++) he += vc[p] * vc[p] / hsq[p];
  he = sqrt(he) / 2.0;
  const double hinv = he == 0.0 ? 0.0 : 1.0 / he;
  out[0] = s * hinv;
#pragma unroll
  for (int b = 0; b < DIM; b++) {
    const double dh = hsq[b] != 0.0 ? vc[b] * hinv / 4.0 / hsq[b] : 0.0;
    out[1 + b] = he != 0.0 ? s * (-dh / he / he) : 0.0;
  }
}

// ---------------------------------------------------------------------------
// QUAD9 element matrices on the matrix cores, four elements per workgroup.
//
// The elements' maps, gradients, fields and residuals are worked out by the
// whole workgroup (a thread per element and point, node or row: one element
// would leave most of a wave idle) and staged in LDS; then each wave takes one
// element, whose node-pair blocks are sums of products E(X, w, Y)[i][j] =
// sum_q X[q][i] w[q] Y[q][j] of 9 x 9 operand tables (the same terms as the
// HEX27 kernel below), one v_mfma_f64_16x16x4f64 tile each (nodes padded to
// 16, the nine points to three k-steps of 4).  The wave writes its element's matrix
// before Dirichlet rows (kel), residual (re) and, with
// PSPG and energy, the continuity x temperature entries (ct); k_gather sums
// them into the MSR rows.  All elements are one launch.
// Bound by the element matrices' traffic for large meshes and by the chain of
// phases (about 10 us) for small ones.  Measured (assembly of 128 x 128
// shear-thinning elements with energy, FP64): 206 us with k_gather
// against 406 with four coloured launches of a workgroup per element, a
// thread per node pair and += through the element-to-nonzero map; 16 x 16
// cavity 60 us against 100.
typedef double d4v __attribute__((ext_vector_type(4)));

// entry r of n tiles to n neighbouring places, 16 bytes at a time
template <int n>
__device__ inline void put_cols(double *p, const d4v *D, int r) {
  typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
#pragma unroll
  for (int b = 0; b < n / 2 * 2; b += 2) *(Two *)(p + b) = Two{D[b][r], D[b + 1][r]};
  if constexpr (n & 1) p[n - 1] = D[n - 1][r];
}

template <int EN>
struct Quad9Lds {  // one element
  static constexpr int NVE = 9, KP = 12, LD = 16, NV = 2 + EN, NSP = STab<2>::NSP;
  double x[2][NVE], u[NV][NVE], ud[NV][NVE], p[3];
  double B[NVE][2][2];
  double dA[KP];
  double G[2][KP][LD];
  double v[KP][2], gv[KP][2][2], gT[KP][2];  // gv[p][a] = d v_a / d x_p
  double P[KP], mu[KP], dmu[KP], div[KP], Td[KP], f[KP][2], vd[KP][2];
  double ps[KP][2];  // PSPG: tau dA (rho v_dot + rho v.grad v + grad P - f)
  double su[4];      // energy SUPG: s/h, s d(1/h)/d vc_b
  double qw[GM_QS_MAX][NSP], qh[GM_QS_MAX][NSP];  // QSIDE / QCONV: w |J_s| (q + h (T_c - T)), w |J_s| h
  int qsd[GM_QS_MAX];
};

template <int EN, int VISC>
__global__ __launch_bounds__(256, EN && VISC ? 4 : 5) void k_elem2(FillArgs A, int num_elems) {
  constexpr int DIM = 2, NVE = 9, NQ = 9, NP = 3, NV = DIM + EN, NVE2 = NVE * NVE;
  constexpr int KP = 12, LD = 16, NL = NV * NVE + NP;
  using T = Tab<2>;
  constexpr int NSP = STab<2>::NSP, SREC = STab<2>::REC;
  __shared__ double s_Phi[KP][LD], s_dphi[NQ][NVE][DIM], s_psi[NQ][NP], s_wt[NQ];
  __shared__ Quad9Lds<EN> s_el[4];
  const double *__restrict__ tb = A.tables;
  for (int t = threadIdx.x; t < KP * LD; t += 256) {
    const int q = t / LD, i = t - q * LD;
    s_Phi[q][i] = (q < NQ && i < NVE) ? tb[T::PHI + q * NVE + i] : 0.0;
  }
  for (int t = threadIdx.x; t < NQ * NVE * DIM; t += 256) (&s_dphi[0][0][0])[t] = tb[T::DPHI + t];
  if (threadIdx.x < NQ * NP) (&s_psi[0][0])[threadIdx.x] = tb[T::PSI + threadIdx.x];
  else if (threadIdx.x >= 64 && threadIdx.x < 64 + NQ) s_wt[threadIdx.x - 64] = tb[T::WT + threadIdx.x - 64];
  const int tid = threadIdx.x, e0 = xcd_block() * 4, ne = min(4, num_elems - e0);

  // 1. gather, a thread per element and node (the centroid carries the pressures)
  if (tid < ne * NVE) {
    const int el = tid / NVE, i = tid - el * NVE;
    Quad9Lds<EN> &S = s_el[el];
    const int n = A.conn[(size_t)e0 * NVE + tid];
    const int f = A.fu[n];
#pragma unroll
    for (int k = 0; k < DIM; k++) S.x[k][i] = A.coor[(size_t)k * A.num_nodes + n];
#pragma unroll
    for (int a = 0; a < NV; a++) {
      const double xv = A.x[f + a];
      S.u[a][i] = xv;
      // xdot as solve_nonlinear_problem forms it after each update (src/rf_solve.c:2848)
      S.ud[a][i] = A.x_old ? A.cmass * (xv - A.x_old[f + a]) - A.cold * A.xdot_old[f + a] : 0.0;
    }
  } else if (tid >= 64 && tid < 64 + ne) {
    const int f = A.fu[A.centroid[e0 + tid - 64]] + NV;
#pragma unroll
    for (int k = 0; k < NP; k++) s_el[tid - 64].p[k] = A.x[f + k];
  }
  __syncthreads();

  // 2. map per point (beer_belly): a thread per element, point and J[i][j]
  if (tid < 36 * ne) {
    const int el = tid / 36, t = tid - el * 36, q = t >> 2, i = (t >> 1) & 1, j = t & 1;
    Quad9Lds<EN> &S = s_el[el];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NVE; k++) s += S.x[j][k] * s_dphi[q][k][i];
    S.B[q][i][j] = s;
  } else if (tid >= 192 && tid < 192 + ne) {
    Quad9Lds<EN> &S = s_el[tid - 192];
    double vc[DIM], su[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < DIM; p++) vc[p] = S.u[p][NVE - 1];
    if (EN && A.supg_e != 0.0) supg_params<DIM>(A.supg_e, S.x, vc, su);
#pragma unroll
    for (int k = 0; k < 4; k++) S.su[k] = su[k];
  } else if (EN && A.qs_ptr && tid >= 196 && tid < 196 + ne * GM_QS_MAX * NSP) {
    // QSIDE (src/bc_integ.c:1518-1519, 2156-2157): w * |surface Jacobian| * q
    // at one surface Gauss point of one side entry; the side's free reference
    // axis gives the tangent, as get_side_info orders it
    // (src/mm_fill_fill.c:3049-3072, 3182-3250)
    const int el = (tid - 196) / (GM_QS_MAX * NSP), t = tid - 196 - el * GM_QS_MAX * NSP;
    const int k = t / NSP, g = t - k * NSP, at = A.qs_ptr[e0 + el] + k;
    if (at < A.qs_ptr[e0 + el + 1]) {
      Quad9Lds<EN> &S = s_el[el];
      const int sd = A.qs_side[at] - 1;
      const double *st = A.stab + (size_t)(sd * NSP + g) * SREC;
      const int fr = (sd == 0 || sd == 2) ? 0 : 1;
      double t1[DIM], Tg = 0.0;
#pragma unroll
      for (int j = 0; j < DIM; j++) {
        t1[j] = 0.0;
        for (int i = 0; i < NVE; i++) t1[j] += S.x[j][i] * st[NVE + i * DIM + fr];
      }
      const double *qk = A.qs_q + 3 * at;
      const double wd = st[NVE + NVE * DIM] * sqrt(t1[0] * t1[0] + t1[1] * t1[1]);
      if constexpr (EN)
        for (int j = 0; j < NVE; j++) Tg += st[j] * S.u[DIM][j];
      S.qw[k][g] = wd * (qk[0] + qk[1] * (qk[2] - Tg));
      S.qh[k][g] = wd * qk[1];
      if (g == 0) S.qsd[k] = sd;
    }
  }
  static_assert(196 + 4 * GM_QS_MAX * NSP <= 256, "side entries of four elements in one pass");
  __syncthreads();
  if (tid >= 64 && tid < 64 + ne * KP) {
    const int el = (tid - 64) / KP, q = tid - 64 - el * KP;
    Quad9Lds<EN> &S = s_el[el];
    double dA = 0.0;
    if (q < NQ) {
      const double J00 = S.B[q][0][0], J01 = S.B[q][0][1], J10 = S.B[q][1][0], J11 = S.B[q][1][1];
      const double det = J00 * J11 - J01 * J10;
      S.B[q][0][0] = J11 / det;
      S.B[q][0][1] = -J01 / det;
      S.B[q][1][0] = -J10 / det;
      S.B[q][1][1] = J00 / det;
      if (!(det > 0.0)) *(volatile int *)A.flag = 1;
      dA = det * s_wt[q];
    }
    S.dA[q] = dA;  // the padding points carry no weight
  }
  __syncthreads();

  // 3. physical gradients into the padded operand tables (load_bf_grad)
#pragma unroll 1
  for (int t = tid; t < ne * KP * LD; t += 256) {
    const int el = t / (KP * LD), r = t - el * KP * LD, q = r / LD, i = r - q * LD;
    Quad9Lds<EN> &S = s_el[el];
    double g0 = 0.0, g1 = 0.0;
    if (q < NQ && i < NVE) {
      const double d0 = s_dphi[q][i][0], d1 = s_dphi[q][i][1];
      g0 = S.B[q][0][0] * d0 + S.B[q][0][1] * d1;
      g1 = S.B[q][1][0] * d0 + S.B[q][1][1] * d1;
    }
    S.G[0][q][i] = g0;
    S.G[1][q][i] = g1;
  }
  __syncthreads();

  // 4. fields at the points (load_fv, load_fv_grads): a thread per element,
  // point and variable
  if (tid < ne * KP * NV) {
    const int el = tid / (KP * NV), r = tid - el * KP * NV, q = r / NV, a = r - q * NV;
    Quad9Lds<EN> &S = s_el[el];
    double s = 0.0, sd = 0.0, g0 = 0.0, g1 = 0.0;
    if (q < NQ) {
#pragma unroll 3
      for (int k = 0; k < NVE; k++) {
        const double ua = S.u[a][k], ph = s_Phi[q][k];
        s += ua * ph;
        sd += S.ud[a][k] * ph;
        g0 += ua * S.G[0][q][k];
        g1 += ua * S.G[1][q][k];
      }
    }
    if (a < DIM) {
      S.v[q][a] = s;
      S.vd[q][a] = sd;
      S.gv[q][0][a] = g0;
      S.gv[q][1][a] = g1;
    } else {
      S.f[q][0] = s;  // T, replaced by the body force below
      S.Td[q] = sd;
      S.gT[q][0] = g0;
      S.gT[q][1] = g1;
    }
  }
  __syncthreads();
  if (tid >= 192 && tid < 192 + ne * KP) {
    const int el = (tid - 192) / KP, q = tid - 192 - el * KP;
    Quad9Lds<EN> &S = s_el[el];
    const double Tq = EN ? S.f[q][0] : 0.0;
    double gv[DIM][DIM], v[DIM];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
      v[a] = S.v[q][a];
#pragma unroll
      for (int p = 0; p < DIM; p++) gv[p][a] = S.gv[q][p][a];
    }
    double P = 0.0, mu = A.mu0, dmu = 0.0;
    if (q < NQ)
#pragma unroll
      for (int k = 0; k < NP; k++) P += S.p[k] * s_psi[q][k];
    if constexpr (VISC == 1) {
      // calc_shearrate + carreau_viscosity (src/mm_fill_util.c:4564,
      // src/mm_viscosity.c:1065-1116); the derivative's powers are the
      // viscosity's own over one factor each (1 where the first overflows)
      double gd = 0.0;
#pragma unroll
      for (int a = 0; a < DIM; a++)
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          const double gab = gv[a][b] + gv[b][a];
          gd += gab * gab;
        }
      gd = sqrt(0.5 * fabs(gd));
      const bool nz = fabs(gd) > 1.0e-298;
      const double val2 = nz ? pow(A.lam * gd, A.aexp) : 0.0;
      const double pm = pow(1.0 + val2, (A.nexp - 1.0) / A.aexp);
      mu = A.muinf + (A.mu0 - A.muinf) * pm;
      if (nz) dmu = (A.mu0 - A.muinf) * (A.nexp - 1.0) * pm * (val2 > 1.0e300 ? 1.0 : val2 / (1.0 + val2)) / gd / gd;
    }
    S.P[q] = P;
    S.mu[q] = mu;
    S.dmu[q] = dmu;
    S.div[q] = gv[0][0] + gv[1][1];
    if (!EN) {
      S.Td[q] = 0.0;
      S.gT[q][0] = S.gT[q][1] = 0.0;
    }
    const double wp = A.tau_pspg * S.dA[q];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
      const double f = EN && q < NQ ? A.rho * A.g[a] * (-A.beta * (Tq - A.Tref)) : 0.0;
      double adv = 0.0, gP = 0.0;
#pragma unroll
      for (int p = 0; p < DIM; p++) adv += v[p] * gv[p][a];
      if (q < NQ)
#pragma unroll
        for (int k = 1; k < NP; k++) gP += S.p[k] * S.B[q][a][k - 1];
      S.f[q][a] = f;
      S.ps[q][a] = wp * (A.rho * (adv + S.vd[q][a]) + gP - f);
    }
  }
  __syncthreads();

  const double rho = A.rho, rCp = A.rho * A.Cp, kc = A.kcond;
  const double cm = A.x_old ? A.cmass : 0.0;  // d xdot / d x: the mass-matrix coefficient

  // 5a. residual rows, a thread per element and row
  if (tid < ne * NL) {
    const int el = tid / NL, t = tid - el * NL, e = e0 + el;
    const Quad9Lds<EN> &S = s_el[el];
    double R = 0.0;
    if (t < NV * NVE) {
      const int a = t / NVE, i = t - a * NVE;
      if (a < DIM) {
#pragma unroll 1
        for (int q = 0; q < NQ; q++) {
          const double ph = s_Phi[q][i];
          double adv = 0.0, dif = 0.0;
#pragma unroll
          for (int p = 0; p < DIM; p++) {
            adv += S.v[q][p] * S.gv[q][p][a];
            const double Pi_ap = (a == p ? -S.P[q] : 0.0) + S.mu[q] * (S.gv[q][a][p] + S.gv[q][p][a]);
            dif += S.G[p][q][i] * Pi_ap;
          }
          R += S.dA[q] * (-rho * ph * adv - dif + ph * S.f[q][a] - rho * ph * S.vd[q][a]);
        }
      } else {
#pragma unroll 1
        for (int q = 0; q < NQ; q++) {
          const double ph = s_Phi[q][i];
          double adv = 0.0, dif = 0.0, vgi = 0.0;
#pragma unroll
          for (int p = 0; p < DIM; p++) {
            adv += S.v[q][p] * S.gT[q][p];
            dif += S.G[p][q][i] * S.gT[q][p];
            vgi += S.v[q][p] * S.G[p][q][i];
          }
          R += S.dA[q] * (-rCp * (ph + S.su[0] * vgi) * adv - kc * dif + ph * A.hsrc - rCp * ph * S.Td[q]);
        }
        const int nqs = A.qs_ptr ? A.qs_ptr[e + 1] - A.qs_ptr[e] : 0;
        for (int k = 0; k < nqs; k++)
          for (int g = 0; g < NSP; g++) R += S.qw[k][g] * A.stab[(size_t)(S.qsd[k] * NSP + g) * SREC + i];
      }
    } else {
      const int k = t - NV * NVE;
#pragma unroll 1
      for (int q = 0; q < NQ; q++) R += S.dA[q] * s_psi[q][k] * S.div[q];
      if (A.tau_pspg != 0.0 && k > 0)
#pragma unroll 1
        for (int q = 0; q < NQ; q++)
#pragma unroll
          for (int a = 0; a < DIM; a++) R += S.B[q][a][k - 1] * S.ps[q][a];
    }
    A.re[(size_t)e0 * NL + tid] = R;
  }
  if (A.resid_only) return;

  // from here on a wave per element
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), e = e0 + w;
  if (w >= ne) return;
  const Quad9Lds<EN> &S = s_el[w];
  const double sw = S.su[0];
  const int qs0 = EN && A.qs_ptr ? A.qs_ptr[e] : 0;
  const int nqs = EN && A.qs_ptr ? A.qs_ptr[e + 1] - qs0 : 0;
  double *__restrict__ ke = A.kel + (size_t)e * A.E;

  // 5b. nodal blocks: the lane's rows i = kk + 4 r and column j; operands at node j
  const int j = lane & 15, kk = lane >> 4;
#define GM_MFMA64(a, b, c) __builtin_amdgcn_mfma_f64_16x16x4f64((a), (b), (c), 0, 0, 0)
  const d4v z = {0.0, 0.0, 0.0, 0.0};
  auto store = [&](int a, const d4v *D) {  // block row a
    if (j >= NVE) return;
#pragma unroll
    for (int r = 0; r < 3; r++) {
      const int i = kk + 4 * r;
      if (i < NVE) put_cols<NV>(ke + (a * NVE2 + i * NVE + j) * NV, D, r);
    }
  };
  // shared products: E(phi, dA, phi), and folded into the diagonal blocks
  // E(phi, dA, v.G) and sum_p E(G_p, dA, G_p) (times mu, times k)
  d4v A1 = z, Dm = z, Tt = z;
  {
    d4v Dadv = z, L1 = z, Lmu = z;
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      const double dA = S.dA[q], ph = s_Phi[q][j], g0 = S.G[0][q][j], g1 = S.G[1][q][j];
      const double vg = S.v[q][0] * g0 + S.v[q][1] * g1;
      A1 = GM_MFMA64(ph * dA, ph, A1);
      Dadv = GM_MFMA64(ph * dA, vg, Dadv);
      L1 = GM_MFMA64(g0 * dA, g0, L1);
      if constexpr (VISC == 1) Lmu = GM_MFMA64(g0 * dA * S.mu[q], g0, Lmu);
      L1 = GM_MFMA64(g1 * dA, g1, L1);
      if constexpr (VISC == 1) Lmu = GM_MFMA64(g1 * dA * S.mu[q], g1, Lmu);
    }
    if constexpr (VISC == 0) Lmu = A.mu0 * L1;
    Dm = -(rho * Dadv + Lmu + (rho * cm) * A1);
    if constexpr (EN) Tt = -(rCp * Dadv + kc * L1 + (rCp * cm) * A1);
  }
#pragma unroll 1
  for (int a = 0; a < DIM; a++) {
    d4v J[NV];
#pragma unroll
    for (int b = 0; b < DIM; b++) J[b] = z;
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      const double dA = S.dA[q], ph = s_Phi[q][j], g[DIM] = {S.G[0][q][j], S.G[1][q][j]};
      const double ga = S.G[a][q][j], wmu = -dA * (VISC ? S.mu[q] : A.mu0);
      double hA = 0.0;
      if constexpr (VISC == 1) {
        // Carreau: (d mu / d gammadot) / gammadot (G_i . gamma_a) (g_j . gamma_b)
#pragma unroll
        for (int p = 0; p < DIM; p++) hA += g[p] * (S.gv[q][a][p] + S.gv[q][p][a]);
        hA *= -dA * S.dmu[q];
      }
#pragma unroll
      for (int b = 0; b < DIM; b++) {
        // advection through d_b v_a, then mu g_j,a G_i,b
        J[b] = GM_MFMA64(ph * (-rho * dA) * S.gv[q][b][a], ph, J[b]);
        J[b] = GM_MFMA64(g[b] * wmu, ga, J[b]);
        if constexpr (VISC == 1) {
          double hB = 0.0;
#pragma unroll
          for (int p = 0; p < DIM; p++) hB += g[p] * (S.gv[q][b][p] + S.gv[q][p][b]);
          J[b] = GM_MFMA64(hA, hB, J[b]);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < DIM; b++) J[b] = a == b ? J[b] + Dm : J[b];
    if constexpr (EN) J[DIM] = (-rho * A.g[a] * A.beta) * A1;
    store(a, J);
  }
  if constexpr (EN) {
    d4v Jb[NV];
#pragma unroll
    for (int b = 0; b < DIM; b++) Jb[b] = z;
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      // (phi_i + sw v.G_i) d_b T + sw (v.grad T) G_b,i: the SUPG weight on
      // the advection and its derivative in v at the column node; and the
      // weight's part of J_TT, -rho Cp sw E(v.G_i dA, v.G_j)
      const double ph = s_Phi[q][j], g[DIM] = {S.G[0][q][j], S.G[1][q][j]};
      const double vg = S.v[q][0] * g[0] + S.v[q][1] * g[1];
      const double wt = -rCp * S.dA[q], vgT = S.v[q][0] * S.gT[q][0] + S.v[q][1] * S.gT[q][1];
#pragma unroll
      for (int b = 0; b < DIM; b++)
        Jb[b] = GM_MFMA64(wt * ((ph + sw * vg) * S.gT[q][b] + sw * vgT * g[b]), ph, Jb[b]);
      if (sw != 0.0) Tt = GM_MFMA64(wt * sw * vg, vg, Tt);
    }
    if (sw != 0.0 && j == NVE - 1) {
      // d(1/h)/dv at the last local node: -rho Cp s_b sum_q dA (v.grad T) v_b G_b,i
#pragma unroll
      for (int r = 0; r < 3; r++) {
        const int i = kk + 4 * r;
        if (i >= NVE) continue;
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          double c = 0.0;
#pragma unroll 1
          for (int q = 0; q < NQ; q++)
            c += S.dA[q] * (S.v[q][0] * S.gT[q][0] + S.v[q][1] * S.gT[q][1]) * S.v[q][b] * S.G[b][q][i];
          Jb[b][r] -= rCp * S.su[1 + b] * c;
        }
      }
    }
    // QCONV: -h w |surface Jacobian| phi_i phi_j over the element's sides
    for (int k = 0; k < nqs; k++) {
      if (A.qs_q[3 * (qs0 + k) + 1] == 0.0 || j >= NVE) continue;
      for (int g = 0; g < NSP; g++) {
        const double *st = A.stab + (size_t)(S.qsd[k] * NSP + g) * SREC;
#pragma unroll
        for (int r = 0; r < 3; r++)
          if (kk + 4 * r < NVE) Tt[r] -= S.qh[k][g] * st[kk + 4 * r] * st[j];
      }
    }
    Jb[DIM] = Tt;
    store(DIM, Jb);
  }
#undef GM_MFMA64

  // 5c. momentum x pressure (J_m_P): int grad_a phi_i psi_k dA; 5d. continuity
  // x velocity (J_c_v): int psi_k grad_b phi_j dA, plus PSPG's
  // tau rho [phi_j grad psi_k . d_b v + grad_b psi_k (v.grad phi_j + c phi_j)]
  // and continuity x temperature tau rho beta (grad psi_k . g) phi_j
  const bool ps = A.tau_pspg != 0.0;
  if (lane < 2 * NVE * NP) {
    const bool mp = lane < NVE * NP;
    const int t = mp ? lane : lane - NVE * NP;
    const int k = mp ? t % NP : t / NVE, i = mp ? t / NP : t % NVE;
    double acc[DIM] = {0.0, 0.0}, accT = 0.0;
#pragma unroll 3
    for (int q = 0; q < NQ; q++) {
      const double wq = S.dA[q] * s_psi[q][k];
#pragma unroll
      for (int a = 0; a < DIM; a++) acc[a] += wq * S.G[a][q][i];
    }
    if (ps && !mp && k > 0) {
#pragma unroll 1
      for (int q = 0; q < NQ; q++) {
        const double wp = A.tau_pspg * S.dA[q] * rho, phj = s_Phi[q][i];
        double vgj = 0.0, gk[DIM], gkg = 0.0;
#pragma unroll
        for (int p = 0; p < DIM; p++) {
          vgj += S.v[q][p] * S.G[p][q][i];
          gk[p] = S.B[q][p][k - 1];
          gkg += gk[p] * A.g[p];
        }
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          double gv = 0.0;
#pragma unroll
          for (int a = 0; a < DIM; a++) gv += gk[a] * S.gv[q][b][a];
          acc[b] += wp * (phj * gv + gk[b] * (vgj + cm * phj));
        }
        accT += wp * A.beta * gkg * phj;
      }
    }
#pragma unroll
    for (int a = 0; a < DIM; a++) ke[(mp ? A.off_mp : A.off_cv) + a * NVE * NP + t] = acc[a];
    if (EN && ps && !mp) A.ct[(size_t)e * NP * NVE + t] = accT;
  }
  // 5e. continuity x pressure: zero for Galerkin Q2-P1; PSPG adds
  // tau grad psi_k . grad psi_l
  if (lane < NP * NP) {
    const int k = lane / NP, k2 = lane - k * NP;
    double acc = 0.0;
    if (ps && k > 0 && k2 > 0)
#pragma unroll 1
      for (int q = 0; q < NQ; q++)
        acc += A.tau_pspg * S.dA[q] *
               (S.B[q][0][k - 1] * S.B[q][0][k2 - 1] + S.B[q][1][k - 1] * S.B[q][1][k2 - 1]);
    ke[A.off_cp + lane] = acc;
  }
}

// ---------------------------------------------------------------------------
// HEX27 element matrices on the matrix cores.
//
// One workgroup (four waves) per element, all elements in one launch.  Every
// node-pair block of the element Jacobian is a sum of products
//   E(X, w, Y)[i][j] = sum_q X[q][i] w[q] Y[q][j]
// of 27 x 27 operand tables (X, Y in {phi, d phi / d x_p}, weights from the
// fields), computed with v_mfma_f64_16x16x4f64 on the 27 x 27 node-pair
// matrix padded to 32 x 32 (two 16-wide tiles per side, one tile per wave)
// and 27 quadrature points padded to 28 (seven k-steps).  Per block (a, b),
// with c = d xdot / d x (transient), mu constant or Carreau mu(q):
//   J_ab = E(phi, -rho dA d_b v_a, phi) - E(G_b, mu dA, G_a)
//          - delta_ab [rho E(phi, dA, v.G) + sum_p E(G_p, mu dA, G_p) + rho c E(phi, dA, phi)]
//          - E(H_a, c_mu dA, H_b)           (Carreau: H_a = sum_p G_p gamma_ap,
//                                            c_mu = (d mu / d gammadot) / gammadot)
//   J_aT = -rho g_a beta E(phi, dA, phi),   J_Ta = E(phi, -rho Cp dA d_a T, phi)
//   J_TT = -rho Cp E(phi, dA, v.G) - k sum_p E(G_p, dA, G_p) - rho Cp c E(phi, dA, phi)
// (the terms of src/mm_fill_momentum.c:1564-1735, 746-915 and
// src/mm_fill_energy.c:425-487, 620-690 regrouped as products over q).
// MFMA lane layout (checked on the device): lane l supplies A[l%16][l/16]
// and B[l/16][l%16] and holds D[l/16 + 4r][l%16], r = 0..3 (rows interleaved).
//
// The products that are not node by node ride along.  The state at the points
// is one product of the reference tables {d phi / d xi_r, phi} with the nodes'
// (x, u, xdot) as columns.  Columns 27..30 of the padded tables carry the
// residual rows' weights W_a(q) (beside phi) and fluxes -Pi_ap(q) (beside
// d phi / d x_p), so E(phi, dA, phi) + sum_p E(G_p, dA, G_p) holds the
// residual in columns 27 + a; and dA psi_k in those columns of the products
// with G_b gives momentum x pressure, whose transpose is continuity x velocity.
//
// The workgroup writes the element's matrix before Dirichlet rows (kel),
// residual (re) and, with PSPG and energy, the continuity x temperature entries
// (ct); k_gather sums them into the MSR rows.
// Bound by the element matrices' bytes (98 KB an element with energy) and the
// 182 products a wave (64 cycles each).  Measured, with k_gather (16^3
// elements with energy, FP64): 430 us against 742 with eight coloured
// launches that staged the state by threads and added into the rows through a
// rank map; 11^3 shear-thinning, FP32 matrix: 194 against 625.

struct NodeCols {  // coordinates as x[a][i] from rows of 16 doubles a node
  const double *p;
  struct Col {
    const double *p;
    __device__ double operator[](int i) const { return p[i * 16]; }
  };
  __device__ Col operator[](int a) const { return Col{p + a}; }
};

template <int EN, int VISC>
__global__ __launch_bounds__(256, 4) void k_elem3(FillArgs A) {
  constexpr int DIM = 3, NVE = 27, NQ = 27, NP = 4, NV = DIM + EN, NVE2 = NVE * NVE;
  constexpr int KP = 28, LD = 32, NL = NV * NVE + NP, NCOL = DIM + 2 * NV, NG = (KP * LD + 255) / 256;
  using T = Tab<3>;
  constexpr int NSP = STab<3>::NSP, SREC = STab<3>::REC;
  const int e = xcd_block(), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kk = lane >> 4;
  const double *__restrict__ tb = A.tables;

  __shared__ double s_nod[KP][16];  // columns x, u, xdot of each node
  __shared__ double s_p[NP];
  __shared__ double s_B[NQ][DIM][DIM];
  __shared__ double s_dA[KP], s_mu[KP], s_dmu[KP], s_wpsi[KP][NP];
  __shared__ double s_Phi[KP][LD];
  __shared__ double s_G[DIM][KP][LD];
  __shared__ double s_v[KP][DIM];
  __shared__ double s_gv[KP][DIM][DIM];  // gv[p][a] = d v_a / d x_p
  __shared__ double s_gT[KP][DIM];
  __shared__ double s_m[NQ][DIM];  // PSPG: rho v_dot + rho v.grad v + grad P - f
  __shared__ double s_rk[2][NP];
  __shared__ double s_su[4];  // energy SUPG: s/h, s d(1/h)/d vc_b
  __shared__ double s_qw[GM_QS_MAX][NSP], s_qh[GM_QS_MAX][NSP];
  __shared__ int s_qsd[GM_QS_MAX];
  // d(column)/d(xi_r) (r < 3) and the column's value (r = 3) at the points,
  // until the gradients take the space
  double(*s_F)[NQ][12] = (double(*)[NQ][12])&s_G[0][0][0];
  static_assert(4 * NQ * 12 <= DIM * KP * LD && NCOL <= 12, "point fields fit the gradient table");
#define GM_MFMA64(a, b, c) __builtin_amdgcn_mfma_f64_16x16x4f64((a), (b), (c), 0, 0, 0)
  const d4v z = {0.0, 0.0, 0.0, 0.0};
  const int qs0 = EN && A.qs_ptr ? A.qs_ptr[e] : 0;
  const int nqs = EN && A.qs_ptr ? A.qs_ptr[e + 1] - qs0 : 0;

  // 1. gather: 32 threads per column, node by node; this wave's reference
  // table (operand of step 2) and this thread's share of the others
  {
    const int k = tid & 31, c = tid >> 5;
    if (c < DIM + NV) {
      double v = 0.0, vd = 0.0;
      if (k < NVE) {
        const int n = A.conn[(size_t)e * NVE + k];
        if (c < DIM) v = A.coor[(size_t)c * A.num_nodes + n];
        else {
          const int g = A.fu[n] + c - DIM;
          v = A.x[g];
          // xdot as solve_nonlinear_problem forms it after each update (src/rf_solve.c:2848)
          if (A.x_old) vd = A.cmass * (v - A.x_old[g]) - A.cold * A.xdot_old[g];
        }
      }
      if (k < KP) {
        s_nod[k][c] = v;
        if (c >= DIM) s_nod[k][c + NV] = vd;
      }
    } else if (c == 7 && k < NP) {
      s_p[k] = A.x[A.fu[A.centroid[e]] + NV + k];
    }
  }
  double ref[2][KP / 4], dph[NG][DIM];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int s = 0; s < KP / 4; s++) {
      const int q = 16 * t + r16, k = 4 * s + kk;
      ref[t][s] = q < NQ && k < NVE ? tb[wave < 3 ? T::DPHI + (q * NVE + k) * DIM + wave : T::PHI + q * NVE + k] : 0.0;
    }
#pragma unroll
  for (int n = 0; n < NG; n++) {
    const int t = tid + 256 * n, q = t / LD, i = t - q * LD;
    const bool in = q < NQ && i < NVE;
#pragma unroll
    for (int r = 0; r < DIM; r++) dph[n][r] = in ? tb[T::DPHI + (q * NVE + i) * DIM + r] : 0.0;
    if (q < KP) s_Phi[q][i] = in ? tb[T::PHI + q * NVE + i] : 0.0;
  }
  __syncthreads();

  // 2. the columns at the points: wave w takes table w
#pragma unroll
  for (int t = 0; t < 2; t++) {
    d4v D = z;
#pragma unroll
    for (int s = 0; s < KP / 4; s++) D = GM_MFMA64(ref[t][s], s_nod[4 * s + kk][r16], D);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int q = 16 * t + kk + 4 * r;
      if (q < NQ && r16 < NCOL) s_F[wave][q][r16] = D[r];
    }
  }
  if (EN && tid == 255) {
    double vc[DIM], su[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < DIM; p++) vc[p] = s_nod[NVE - 1][DIM + p];
    if (A.supg_e != 0.0) supg_params<DIM>(A.supg_e, NodeCols{&s_nod[0][0]}, vc, su);
#pragma unroll
    for (int k = 0; k < 4; k++) s_su[k] = su[k];
  } else if (EN && tid < nqs * NSP) {
    // QSIDE (src/bc_integ.c:1518-1519, 2156-2157): w |surface Jacobian| q at
    // one surface Gauss point of one side entry
    const int k = tid / NSP, g = tid - k * NSP;
    const int sd = A.qs_side[qs0 + k] - 1;
    const double *st = A.stab + (size_t)(sd * NSP + g) * SREC;
    const int ax = (sd == 0 || sd == 2) ? 1 : (sd == 1 || sd == 3) ? 0 : 2;
    const int fr[2] = {ax == 0 ? 1 : 0, ax == 2 ? 1 : 2};
    double t1[DIM], tt2[DIM];
#pragma unroll
    for (int j = 0; j < DIM; j++) {
      t1[j] = 0.0;
      tt2[j] = 0.0;
#pragma unroll 1
      for (int i = 0; i < NVE; i++) {
        t1[j] += s_nod[i][j] * st[NVE + i * DIM + fr[0]];
        tt2[j] += s_nod[i][j] * st[NVE + i * DIM + fr[1]];
      }
    }
    const double c0 = t1[1] * tt2[2] - t1[2] * tt2[1], c1 = t1[2] * tt2[0] - t1[0] * tt2[2],
                 c2 = t1[0] * tt2[1] - t1[1] * tt2[0];
    const double *qk = A.qs_q + 3 * (qs0 + k);
    const double wd = st[NVE + NVE * DIM] * sqrt(c0 * c0 + c1 * c1 + c2 * c2);
    double Tg = 0.0;
#pragma unroll 1
    for (int j = 0; j < NVE; j++) Tg += st[j] * s_nod[j][2 * DIM];
    s_qw[k][g] = wd * (qk[0] + qk[1] * (qk[2] - Tg));
    s_qh[k][g] = wd * qk[1];
    if (g == 0) s_qsd[k] = sd;
  }
  static_assert(GM_QS_MAX * NSP <= 255, "a thread per surface point");
  __syncthreads();

  // 3. map (beer_belly) and physical gradients of the fields (load_fv,
  // load_fv_grads): a thread per point and variable, each forming the inverse
  const int pq = tid >> 2, pa = tid & 3;
  const bool point = pq < NQ;
  double g[DIM] = {0.0, 0.0, 0.0}, v[DIM] = {0.0, 0.0, 0.0}, uda = 0.0, Tq = 0.0, dA = 0.0;
  if (point) {
    const int q = pq;
    double J[DIM][DIM], B[DIM][DIM];
#pragma unroll
    for (int i = 0; i < DIM; i++)
#pragma unroll
      for (int j = 0; j < DIM; j++) J[i][j] = s_F[i][q][j];
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[2][0] * J[1][2]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[2][0] * J[1][1]);
    B[0][0] = (J[1][1] * J[2][2] - J[2][1] * J[1][2]) / det;
    B[0][1] = -(J[0][1] * J[2][2] - J[2][1] * J[0][2]) / det;
    B[0][2] = (J[0][1] * J[1][2] - J[1][1] * J[0][2]) / det;
    B[1][0] = -(J[1][0] * J[2][2] - J[2][0] * J[1][2]) / det;
    B[1][1] = (J[0][0] * J[2][2] - J[2][0] * J[0][2]) / det;
    B[1][2] = -(J[0][0] * J[1][2] - J[1][0] * J[0][2]) / det;
    B[2][0] = (J[1][0] * J[2][1] - J[2][0] * J[1][1]) / det;
    B[2][1] = -(J[0][0] * J[2][1] - J[2][0] * J[0][1]) / det;
    B[2][2] = (J[0][0] * J[1][1] - J[1][0] * J[0][1]) / det;
    dA = det * tb[T::WT + q];
    if (pa < NV) {
#pragma unroll
      for (int p = 0; p < DIM; p++)
#pragma unroll
        for (int r = 0; r < DIM; r++) g[p] += B[p][r] * s_F[r][q][DIM + pa];
      uda = s_F[3][q][DIM + NV + pa];
    }
#pragma unroll
    for (int p = 0; p < DIM; p++) v[p] = s_F[3][q][DIM + p];
    if constexpr (EN) Tq = s_F[3][q][2 * DIM];
    if (pa == 0) {
      if (!(det > 0.0)) *(volatile int *)A.flag = 1;
#pragma unroll
      for (int p = 0; p < DIM; p++) {
        s_v[q][p] = v[p];
#pragma unroll
        for (int r = 0; r < DIM; r++) s_B[q][p][r] = B[p][r];
      }
      s_dA[q] = dA;
    }
  }
  if (pq < KP) {  // zeros at the padding point
#pragma unroll
    for (int p = 0; p < DIM; p++) {
      if (pa < DIM) s_gv[pq][p][pa] = g[p];
      else s_gT[pq][p] = g[p];
      if (pq == NQ) s_v[NQ][p] = 0.0;
    }
    if (pq == NQ) s_dA[NQ] = s_mu[NQ] = s_dmu[NQ] = s_wpsi[NQ][pa] = 0.0;
  }
  __syncthreads();

  // 4. physical gradients of the basis into the padded tables (load_bf_grad);
  // viscosity, stress and sources at the points into columns 27 + a
#pragma unroll
  for (int n = 0; n < NG; n++) {
    const int t = tid + 256 * n, q = t / LD, i = t - q * LD;
    if (q >= KP || (i >= NVE && i < NVE + NV && q < NQ)) continue;
#pragma unroll
    for (int p = 0; p < DIM; p++) {
      double s = 0.0;
      if (q < NQ && i < NVE) {
#pragma unroll
        for (int r = 0; r < DIM; r++) s += s_B[q][p][r] * dph[n][r];
      }
      s_G[p][q][i] = s;
    }
  }
  const double rho = A.rho, rCp = A.rho * A.Cp, kc = A.kcond;
  const double cm = A.x_old ? A.cmass : 0.0;
  const bool ps = A.tau_pspg != 0.0;
  if (tid < 128) {
    double ck = 0.0;
    if (point) {
      const int q = pq;
      double mu = A.mu0, dmu = 0.0;
      if constexpr (VISC == 1) {
        // calc_shearrate + carreau_viscosity (src/mm_fill_util.c:4564,
        // src/mm_viscosity.c:1065-1116)
        double gd = 0.0;
#pragma unroll
        for (int a = 0; a < DIM; a++)
#pragma unroll
          for (int b = 0; b < DIM; b++) {
            const double gab = s_gv[q][a][b] + s_gv[q][b][a];
            gd += gab * gab;
          }
        gd = sqrt(0.5 * fabs(gd));
        const bool nz = fabs(gd) > 1.0e-298;
        const double val2 = nz ? pow(A.lam * gd, A.aexp) : 0.0;
        const double pm = pow(1.0 + val2, (A.nexp - 1.0) / A.aexp);
        mu = A.muinf + (A.mu0 - A.muinf) * pm;
        // d mu / d gammadot / gammadot; lam^a gd^(a-1) = val2 / gd, and
        // val2 / (1 + val2) is 1 where val2 overflows
        if (nz) dmu = (A.mu0 - A.muinf) * (A.nexp - 1.0) * pm * (val2 > 1.0e300 ? 1.0 : val2 / (1.0 + val2)) / gd / gd;
      }
      double P = 0.0;
#pragma unroll
      for (int k = 0; k < NP; k++) P += s_p[k] * tb[T::PSI + q * NP + k];
      double adv = 0.0;
#pragma unroll
      for (int p = 0; p < DIM; p++) adv += v[p] * g[p];
      if (pa < DIM) {
        const double f = EN ? rho * A.g[pa] * (-A.beta * (Tq - A.Tref)) : 0.0;
        s_Phi[q][NVE + pa] = f - rho * (adv + uda);
#pragma unroll
        for (int p = 0; p < DIM; p++)
          s_G[p][q][NVE + pa] = (pa == p ? P : 0.0) - mu * (g[p] + s_gv[q][pa][p]);
        if (ps) {
          double gP = 0.0;
#pragma unroll
          for (int l = 1; l < NP; l++) gP += s_p[l] * s_B[q][pa][l - 1];
          s_m[q][pa] = rho * (adv + uda) + gP - f;
        }
      } else if constexpr (EN) {
        s_Phi[q][NVE + DIM] = A.hsrc - rCp * (adv + uda);
#pragma unroll
        for (int p = 0; p < DIM; p++) s_G[p][q][NVE + DIM] = -kc * g[p] - rCp * s_su[0] * adv * v[p];
      }
      if (pa == 0) {
        s_mu[q] = mu;
        s_dmu[q] = dmu;
      }
      const double wp = dA * tb[T::PSI + q * NP + pa];
      s_wpsi[q][pa] = wp;
      ck = wp * (s_gv[q][0][0] + s_gv[q][1][1] + s_gv[q][2][2]);
    }
    // continuity residual: psi_k div v over this wave's points
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) ck += __shfl_xor(ck, o);
    if (lane < NP) s_rk[wave][lane] = ck;
  }
  __syncthreads();

  // 5a. shared products: E(phi, dA, phi), E(phi, dA, v.G), sum_p E(G_p, dA,
  // G_p) and (Carreau) its mu-weighted form; the residual in columns 27 + a.
  // Wave w: rows 16 (w >> 1) .. +15, columns 16 (w & 1) .. +15 of every block
  const int i0 = 16 * (wave >> 1), ii = i0 + r16;  // row operand (A)
  const int j = 16 * (wave & 1) + r16;             // column operand (B) and column
  const bool node = j < NVE;
  double *__restrict__ re = A.re + (size_t)e * NL;
  double *__restrict__ K = A.kel + (size_t)e * A.E;
  d4v A1 = z, Lp[DIM] = {z, z, z}, Dadv = z, Lmu = z;
  if (!A.resid_only) {
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      const double dAq = s_dA[q], phA = s_Phi[q][ii] * dAq;
      double vB = 0.0;
#pragma unroll
      for (int p = 0; p < DIM; p++) vB += s_v[q][p] * s_G[p][q][j];
      A1 = GM_MFMA64(phA, s_Phi[q][j], A1);
      Dadv = GM_MFMA64(phA, vB, Dadv);
#pragma unroll
      for (int p = 0; p < DIM; p++) {
        const double gA = s_G[p][q][ii] * dAq, gB = s_G[p][q][j];
        Lp[p] = GM_MFMA64(gA, gB, Lp[p]);
        if constexpr (VISC == 1) Lmu = GM_MFMA64(gA * s_mu[q], gB, Lmu);
      }
    }
  } else if (wave & 1) {
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      const double dAq = s_dA[q];
      A1 = GM_MFMA64(s_Phi[q][ii] * dAq, s_Phi[q][j], A1);
#pragma unroll
      for (int p = 0; p < DIM; p++) Lp[p] = GM_MFMA64(s_G[p][q][ii] * dAq, s_G[p][q][j], Lp[p]);
    }
  }
  const d4v L1 = Lp[0] + Lp[1] + Lp[2];
  if (j >= NVE && j < NVE + NV) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + kk + 4 * r;
      if (i >= NVE) continue;
      double R = A1[r] + L1[r];
      if (EN && j == NVE + DIM)
        for (int k = 0; k < nqs; k++)
#pragma unroll 1
          for (int s = 0; s < NSP; s++) R += s_qw[k][s] * A.stab[(size_t)(s_qsd[k] * NSP + s) * SREC + i];
      re[(j - NVE) * NVE + i] = R;
    }
  }
  if (tid < NP) {
    double R = s_rk[0][tid] + s_rk[1][tid];
    if (ps && tid > 0) {
      // PSPG: grad psi_k . tau (rho v_dot + rho v.grad v + grad P - f) dA
#pragma unroll 1
      for (int q = 0; q < NQ; q++) {
        double r = 0.0;
#pragma unroll
        for (int a = 0; a < DIM; a++) r += s_B[q][a][tid - 1] * s_m[q][a];
        R += A.tau_pspg * s_dA[q] * r;
      }
    }
    re[NV * NVE + tid] = R;
  }
  if (A.resid_only) return;

  // 5b. nodal blocks: rows i0 + kk + 4 r, column j
  auto store = [&](int a, const d4v *D) {  // block row a
    double *__restrict__ k = K + (size_t)(a * NVE2 + j) * NV;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + kk + 4 * r;
      if (i < NVE && node) put_cols<NV>(k + i * NVE * NV, D, r);
    }
  };
  if constexpr (VISC == 0) Lmu = A.mu0 * L1;
  const d4v Dm = -(rho * Dadv + Lmu + (rho * cm) * A1);
  d4v Tt = -(rCp * Dadv + kc * L1 + (rCp * cm) * A1);
#pragma unroll 1
  for (int a = 0; a < DIM; a++) {
    d4v J[NV];
#pragma unroll
    for (int b = 0; b < DIM; b++) J[b] = z;
#pragma unroll 1
    for (int q = kk; q < KP; q += 4) {
      const double dAq = s_dA[q], phA = s_Phi[q][ii] * (-rho * dAq), phB = node ? s_Phi[q][j] : 0.0;
      double gA[DIM];
#pragma unroll
      for (int b = 0; b < DIM; b++) gA[b] = s_G[b][q][ii];
      // columns 27 + k: dA psi_k, momentum x pressure
      const double gB = node ? s_G[a][q][j] * (-dAq * (VISC ? s_mu[q] : A.mu0)) : s_wpsi[q][(j - NVE) & 3];
#pragma unroll
      for (int b = 0; b < DIM; b++) J[b] = GM_MFMA64(phA * s_gv[q][b][a], phB, J[b]);
#pragma unroll
      for (int b = 0; b < DIM; b++) J[b] = GM_MFMA64(gA[b], gB, J[b]);
      if constexpr (VISC == 1) {
        // Carreau: (d mu / d gammadot) / gammadot (G_i . gamma_a) (g_j . gamma_b)
        double hA = 0.0;
#pragma unroll
        for (int p = 0; p < DIM; p++) hA += gA[p] * (s_gv[q][a][p] + s_gv[q][p][a]);
        hA *= -dAq * s_dmu[q];
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          double hB = 0.0;
#pragma unroll
          for (int p = 0; p < DIM; p++) hB += s_G[p][q][j] * (s_gv[q][b][p] + s_gv[q][p][b]);
          J[b] = GM_MFMA64(hA, node ? hB : 0.0, J[b]);
        }
      }
    }
    if (a == 0 && j >= NVE && j < NVE + NP) {
      // momentum x pressure (J_m_P): int grad_b phi_i psi_k dA, and its
      // transpose, continuity x velocity (J_c_v)
      const int k = j - NVE;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + kk + 4 * r;
        if (i >= NVE) continue;
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          K[A.off_mp + (b * NVE + i) * NP + k] = J[b][r];
          if (!ps) K[A.off_cv + (b * NP + k) * NVE + i] = J[b][r];
        }
      }
    }
#pragma unroll
    for (int b = 0; b < DIM; b++) J[b] = a == b ? J[b] + Dm : J[b];
    if constexpr (EN) J[DIM] = (-rho * A.g[a] * A.beta) * A1;
    store(a, J);
  }
  if constexpr (EN) {
    const double sw = s_su[0];
    d4v J[NV];
#pragma unroll
    for (int b = 0; b < DIM; b++) J[b] = z;
    if (sw != 0.0) {
#pragma unroll 1
      for (int q = kk; q < KP; q += 4) {
        const double w = -rCp * s_dA[q], phB = s_Phi[q][j];
        // (phi_i + sw v.G_i) d_b T + sw (v.grad T) G_b,i: the SUPG weight on
        // the advection and its derivative in v at the column node; and the
        // weight's part of J_TT, -rho Cp sw E(v.G_i dA, v.G_j)
        double vA = 0.0, vgT = 0.0, vB = 0.0;
#pragma unroll
        for (int p = 0; p < DIM; p++) {
          vA += s_v[q][p] * s_G[p][q][ii];
          vgT += s_v[q][p] * s_gT[q][p];
          vB += s_v[q][p] * s_G[p][q][j];
        }
        const double wi = s_Phi[q][ii] + sw * vA;
#pragma unroll
        for (int b = 0; b < DIM; b++)
          J[b] = GM_MFMA64(w * (wi * s_gT[q][b] + sw * vgT * s_G[b][q][ii]), phB, J[b]);
        Tt = GM_MFMA64(w * sw * vA, vB, Tt);
      }
      if (j == NVE - 1) {
        // d(1/h)/dv at the last local node: -rho Cp s_b sum_q dA (v.grad T) v_b G_b,i
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = i0 + kk + 4 * r;
          if (i >= NVE) continue;
#pragma unroll
          for (int b = 0; b < DIM; b++) {
            double c = 0.0;
#pragma unroll 1
            for (int q = 0; q < NQ; q++) {
              double vgT = 0.0;
#pragma unroll
              for (int p = 0; p < DIM; p++) vgT += s_v[q][p] * s_gT[q][p];
              c += s_dA[q] * vgT * s_v[q][b] * s_G[b][q][i];
            }
            J[b][r] -= rCp * s_su[1 + b] * c;
          }
        }
      }
    } else {
#pragma unroll 1
      for (int q = kk; q < KP; q += 4) {
        const double phA = s_Phi[q][ii] * (-rCp * s_dA[q]), phB = s_Phi[q][j];
#pragma unroll
        for (int b = 0; b < DIM; b++) J[b] = GM_MFMA64(phA * s_gT[q][b], phB, J[b]);
      }
    }
    // QCONV: -h w |surface Jacobian| phi_i phi_j over the element's sides
    for (int k = 0; k < nqs; k++) {
      if (A.qs_q[3 * (qs0 + k) + 1] == 0.0 || !node) continue;
#pragma unroll 1
      for (int s = 0; s < NSP; s++) {
        const double *st = A.stab + (size_t)(s_qsd[k] * NSP + s) * SREC;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = i0 + kk + 4 * r;
          if (i < NVE) Tt[r] -= s_qh[k][s] * st[i] * st[j];
        }
      }
    }
    J[DIM] = Tt;
    store(DIM, J);
  }
#undef GM_MFMA64

  // 5c. PSPG: continuity x velocity gains tau rho [phi_j grad psi_k . d_b v +
  // grad_b psi_k (v.grad phi_j + c phi_j)], continuity x temperature is tau rho
  // beta (grad psi_k . g) phi_j, continuity x pressure tau grad psi_k . grad psi_l
  if (ps)
    for (int t = tid; t < NP * NVE; t += 256) {
      const int k = t / NVE, n = t - k * NVE;
      double acc[DIM] = {0.0, 0.0, 0.0}, accT = 0.0;
#pragma unroll 1
      for (int q = 0; q < NQ; q++) {
        const double w = s_wpsi[q][k];
#pragma unroll
        for (int b = 0; b < DIM; b++) acc[b] += w * s_G[b][q][n];
        if (k == 0) continue;
        const double wp = A.tau_pspg * s_dA[q] * rho, phj = s_Phi[q][n];
        double vg = 0.0, gk[DIM], gkg = 0.0;
#pragma unroll
        for (int p = 0; p < DIM; p++) {
          vg += s_v[q][p] * s_G[p][q][n];
          gk[p] = s_B[q][p][k - 1];
          gkg += gk[p] * A.g[p];
        }
#pragma unroll
        for (int b = 0; b < DIM; b++) {
          double gv = 0.0;
#pragma unroll
          for (int a = 0; a < DIM; a++) gv += gk[a] * s_gv[q][b][a];
          acc[b] += wp * (phj * gv + gk[b] * (vg + cm * phj));
        }
        accT += wp * A.beta * gkg * phj;
      }
#pragma unroll
      for (int b = 0; b < DIM; b++) K[A.off_cv + b * NP * NVE + t] = acc[b];
      if constexpr (EN) A.ct[(size_t)e * NP * NVE + t] = accT;
    }
  if (tid < NP * NP) {
    const int k = tid / NP, k2 = tid - k * NP;
    double acc = 0.0;
    if (ps && k > 0 && k2 > 0)
#pragma unroll 1
      for (int q = 0; q < NQ; q++) {
        double g2 = 0.0;
#pragma unroll
        for (int a = 0; a < DIM; a++) g2 += s_B[q][a][k - 1] * s_B[q][a][k2 - 1];
        acc += A.tau_pspg * s_dA[q] * g2;
      }
    K[A.off_cp + tid] = acc;
  }
}

// Element-to-nonzero map: for every local entry of every element, the MSR
// index of the global (row, column) pair; the diagonal lives at index row.
template <int DIM>
__global__ __launch_bounds__(256) void k_build_e2nz(const int *__restrict__ conn,
                                                    const int *__restrict__ fu,
                                                    const int *__restrict__ centroid,
                                                    const int *__restrict__ bindx, int en,
                                                    long long E, long long off_mp,
                                                    long long off_cv, long long off_cp,
                                                    int *__restrict__ e2nz, int *flag) {
  constexpr int NVE = El<DIM>::NVE, NP = El<DIM>::NP;
  const int NV = DIM + en;
  const int e = blockIdx.x;
  __shared__ int s_f[NVE];
  __shared__ int s_pc;
  if (threadIdx.x < NVE) s_f[threadIdx.x] = fu[conn[(size_t)e * NVE + threadIdx.x]];
  if (threadIdx.x == 0) s_pc = fu[centroid[e]] + DIM + en;
  __syncthreads();
  for (long long idx = threadIdx.x; idx < E; idx += blockDim.x) {
    int row, col;
    if (idx < off_mp) {
      const int blk = (int)(idx / (NVE * NVE)), t = (int)(idx - (long long)blk * NVE * NVE);
      const int a = blk / NV, b = blk - a * NV;
      row = s_f[t / NVE] + a;
      col = s_f[t % NVE] + b;
    } else if (idx < off_cv) {
      const int r = (int)(idx - off_mp);
      const int a = r / (NVE * NP), t = r - a * NVE * NP;
      row = s_f[t / NP] + a;
      col = s_pc + t % NP;
    } else if (idx < off_cp) {
      const int r = (int)(idx - off_cv);
      const int b = r / (NP * NVE), t = r - b * NP * NVE;
      row = s_pc + t / NVE;
      col = s_f[t % NVE] + b;
    } else {
      const int r = (int)(idx - off_cp);
      row = s_pc + r / NP;
      col = s_pc + r % NP;
    }
    int pos;
    if (row == col) {
      pos = row;
    } else {
      int lo = bindx[row], hi = bindx[row + 1] - 1;
      pos = -1;
      while (lo <= hi) {
        const int mid = (lo + hi) >> 1;
        const int v = bindx[mid];
        if (v == col) {
          pos = mid;
          break;
        }
        if (v < col) lo = mid + 1;
        else hi = mid - 1;
      }
      if (pos < 0) atomicOr(&flag[1], 1);
    }
    e2nz[(size_t)e * E + idx] = pos;
  }
}

// Reference basis tables on the host.  QUAD9 closed forms of
// src/rf_shape.c:361-470; HEX27 as products of 1D quadratic Lagrange factors
// (identical to the closed forms of src/rf_shape.c:1105-1460); Gauss points
// ordered as find_stu (src/el_elm_info.c:1748-1823).
static const signed char kHex27[27][3] = {
    {-1, -1, -1}, {1, -1, -1}, {1, 1, -1}, {-1, 1, -1}, {-1, -1, 1}, {1, -1, 1}, {1, 1, 1},
    {-1, 1, 1},   {0, -1, -1}, {1, 0, -1}, {0, 1, -1},  {-1, 0, -1}, {-1, -1, 0}, {1, -1, 0},
    {1, 1, 0},    {-1, 1, 0},  {0, -1, 1}, {1, 0, 1},   {0, 1, 1},   {-1, 0, 1},  {0, 0, 0},
    {0, 0, -1},   {0, 0, 1},   {-1, 0, 0}, {1, 0, 0},   {0, -1, 0},  {0, 1, 0}};
static const signed char kQuad9[9][2] = {{-1, -1}, {1, -1}, {1, 1}, {-1, 1}, {0, -1},
                                        {1, 0},   {0, 1},  {-1, 0}, {0, 0}};

static void lagrange1(int node, double s, double &v, double &dv) {
  if (node < 0) {
    v = -0.5 * s * (1.0 - s);
    dv = -0.5 + s;
  } else if (node > 0) {
    v = 0.5 * s * (1.0 + s);
    dv = 0.5 + s;
  } else {
    v = 1.0 - s * s;
    dv = -2.0 * s;
  }
}

// Q2 basis (QUAD9 / HEX27, Goma local node order) at one reference point.
void gm_q2_basis(int dim, const double *xi, double *phi) {
  const int nve = dim == 2 ? 9 : 27;
  for (int k = 0; k < nve; k++) {
    const signed char *pos = dim == 2 ? kQuad9[k] : kHex27[k];
    double v = 1.0, a, da;
    for (int d = 0; d < dim; d++) {
      lagrange1(pos[d], xi[d], a, da);
      v *= a;
    }
    phi[k] = v;
  }
}

static std::vector<double> make_tables(int dim) {
  const int nve = dim == 2 ? 9 : 27, nq = nve, np = dim + 1;
  std::vector<double> t((size_t)nq * nve + (size_t)nq * nve * dim + (size_t)nq * np + nq);
  double *phi = t.data(), *dphi = phi + nq * nve, *psi = dphi + nq * nve * dim, *wt = psi + nq * np;
  const double F2 = 0.77459666924148340428, w1 = 0.55555555555555555556, w2 = 0.88888888888888888888;
  const double pt[3] = {F2, 0.0, -F2}, ww[3] = {w1, w2, w1};
  for (int q = 0; q < nq; q++) {
    const int is = q % 3, it = (q % 9) / 3, iu = q / 9;
    const double s = pt[is], tt = pt[it], u = dim == 3 ? pt[iu] : 0.0;
    wt[q] = ww[is] * ww[it] * (dim == 3 ? ww[iu] : 1.0);
    for (int k = 0; k < nve; k++) {
      double a, da, b, db, cc = 1.0, dc = 0.0;
      const signed char *pos = dim == 2 ? kQuad9[k] : kHex27[k];
      lagrange1(pos[0], s, a, da);
      lagrange1(pos[1], tt, b, db);
      if (dim == 3) lagrange1(pos[2], u, cc, dc);
      phi[q * nve + k] = a * b * cc;
      dphi[(q * nve + k) * dim + 0] = da * b * cc;
      dphi[(q * nve + k) * dim + 1] = a * db * cc;
      if (dim == 3) dphi[(q * nve + k) * dim + 2] = a * b * dc;
    }
    // P1 discontinuous basis {1, s, t[, u]} (src/mm_fill_util.c:3802-3858, 4205-4276)
    psi[q * np + 0] = 1.0;
    psi[q * np + 1] = s;
    psi[q * np + 2] = tt;
    if (dim == 3) psi[q * np + 3] = u;
  }
  return t;
}

// Side tables (STab layout): the Q2 basis and its reference derivatives at
// the 3 (2D) or 3 x 3 (3D) Gauss points of each side, sides in Exodus order
// (get_side_info, src/mm_fill_fill.c:3049-3072, 3182-3250): the fixed
// reference axis and value of sides 1..2*dim are (t,-1) (s,+1) (t,+1) (s,-1)
// (u,-1) (u,+1); the free axes run in ascending order, the first slowest.
static std::vector<double> make_side_tables(int dim) {
  const int nve = dim == 2 ? 9 : 27, nside = 2 * dim, nsp = dim == 2 ? 3 : 9;
  const int rec = nve + nve * dim + 1;
  static const int axis[6] = {1, 0, 1, 0, 2, 2};
  static const double fixv[6] = {-1.0, 1.0, 1.0, -1.0, -1.0, 1.0};
  const double F2 = 0.77459666924148340428, w1 = 0.55555555555555555556, w2 = 0.88888888888888888888;
  const double gp[3] = {-F2, 0.0, F2}, gw[3] = {w1, w2, w1};
  std::vector<double> t((size_t)nside * nsp * rec);
  for (int sd = 0; sd < nside; sd++) {
    int fr[2], nf = 0;
    for (int a = 0; a < dim; a++)
      if (a != axis[sd]) fr[nf++] = a;
    for (int g = 0; g < nsp; g++) {
      const int g1 = dim == 2 ? g : g / 3, g2 = dim == 2 ? 0 : g % 3;
      double ref[3] = {0.0, 0.0, 0.0};
      ref[axis[sd]] = fixv[sd];
      ref[fr[0]] = gp[g1];
      double w = gw[g1];
      if (dim == 3) {
        ref[fr[1]] = gp[g2];
        w *= gw[g2];
      }
      double *r = t.data() + (size_t)(sd * nsp + g) * rec;
      for (int k = 0; k < nve; k++) {
        const signed char *pos = dim == 2 ? kQuad9[k] : kHex27[k];
        double v[3], dv[3];
        for (int d = 0; d < dim; d++) lagrange1(pos[d], ref[d], v[d], dv[d]);
        double ph = 1.0;
        for (int d = 0; d < dim; d++) ph *= v[d];
        r[k] = ph;
        for (int d = 0; d < dim; d++) {
          double dd = dv[d];
          for (int e = 0; e < dim; e++)
            if (e != d) dd *= v[e];
          r[nve + k * dim + d] = dd;
        }
      }
      r[nve + nve * dim] = w;
    }
  }
  return t;
}

int gm_fill_setup_device(gm_ctx *c) {
  ElemLayout &L = c->lay;
  L.dim = c->dim;
  L.nve = c->nve;
  L.np = c->np;
  L.nv = c->nv;
  L.nq = c->nve;
  const long long nve2 = (long long)L.nve * L.nve;
  L.off_mp = (long long)L.nv * L.nv * nve2;
  L.off_cv = L.off_mp + (long long)L.dim * L.nve * L.np;
  L.off_cp = L.off_cv + (long long)L.dim * L.np * L.nve;
  L.total = L.off_cp + (long long)L.np * L.np;

  std::vector<double> tab = make_tables(c->dim);
  GM_HIP(hipMalloc(&c->d_tables, tab.size() * sizeof(double)));
  GM_HIP(hipMemcpy(c->d_tables, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
  std::vector<double> stab = make_side_tables(c->dim);
  GM_HIP(hipMalloc(&c->d_stab, stab.size() * sizeof(double)));
  GM_HIP(hipMemcpy(c->d_stab, stab.data(), stab.size() * sizeof(double), hipMemcpyHostToDevice));
  return gm_gather_setup(c);
}

// The element-to-nonzero map, which the multigrid's element-block inversions
// read: built when a context becomes a level of a hierarchy.
int gm_e2nz_setup(gm_ctx *c) {
  if (c->d_e2nz) return GM_OK;
  const ElemLayout &L = c->lay;
  int *map = nullptr;
  auto build = [&]() -> int {
    GM_HIP(hipMalloc(&map, (size_t)c->num_elems * L.total * sizeof(int)));
    GM_HIP(hipMemsetAsync(c->d_flag, 0, 4 * sizeof(int), c->stream));
    auto kern = c->dim == 2 ? k_build_e2nz<2> : k_build_e2nz<3>;
    kern<<<c->num_elems, 256, 0, c->stream>>>(c->d_conn, c->d_fu, c->d_centroid, c->d_bindx, c->energy, L.total,
                                              L.off_mp, L.off_cv, L.off_cp, map, c->d_flag);
    GM_HIP(hipGetLastError());
    int flag[4];
    GM_HIP(hipMemcpyAsync(flag, c->d_flag, 4 * sizeof(int), hipMemcpyDeviceToHost, c->stream));
    GM_HIP(hipStreamSynchronize(c->stream));
    if (flag[1]) {
      gm_set_error("element-to-nonzero map: entry missing from the MSR graph");
      return GM_ERR_ARG;
    }
    return GM_OK;
  };
  const int rc = build();
  if (rc) (void)hipFree(map);
  else c->d_e2nz = map;
  return rc;
}

// ct: the continuity x temperature entries are assembled too
static int elem_buffers(gm_ctx *c, bool ct) {
  if (!c->d_re) GM_HIP(hipMalloc(&c->d_re, (size_t)c->num_elems * (c->nv * c->nve + c->np) * sizeof(double)));
  if (ct && !c->d_ct) GM_HIP(hipMalloc(&c->d_ct, (size_t)c->num_elems * c->np * c->nve * sizeof(double)));
  return GM_OK;
}

// The element matrices and residuals of every element, then the rows.
static int assemble(gm_ctx *c, const FillArgs &a, double *resid, double *val, float *val32) {
  const int en = c->energy, vm = c->phys.visc_model;
  const int id = a.resid_only ? GM_K_FILL_RESID : GM_K_FILL;
  // coordinates, connectivity, the state; the element matrices and residuals written
  const double bytes = 8.0 * c->dim * c->num_nodes + 8.0 * c->N + 4.0 * c->nve * c->num_elems +
                       8.0 * c->num_elems * (c->nv * c->nve + c->np + (a.resid_only ? 0.0 : (double)c->lay.total));
  if (c->dim == 2)
    gm_launch(c, id, bytes, en ? (vm ? k_elem2<1, 1> : k_elem2<1, 0>) : (vm ? k_elem2<0, 1> : k_elem2<0, 0>),
              dim3((c->num_elems + 3) / 4), dim3(256), 0, c->stream, a, c->num_elems);
  else
    gm_launch(c, id, bytes, en ? (vm ? k_elem3<1, 1> : k_elem3<1, 0>) : (vm ? k_elem3<0, 1> : k_elem3<0, 0>),
              dim3(c->num_elems), dim3(256), 0, c->stream, a);
  GM_HIP(hipGetLastError());
  const bool mat = !a.resid_only;
  return gm_gather(c, id, c, c->stream, a.kel, en && a.tau_pspg != 0.0 ? a.ct : nullptr, mat && !val32 ? val : nullptr,
                   mat ? val32 : nullptr, c->fill_overwrite, a.re, a.x, resid);
}

int gm_fill_launch(gm_ctx *c, const double *x, double *resid, double *val, float *val32) {
  return gm_fill_launch_ex(c, x, resid, val, val32, 0);
}

int gm_fill_launch_ex(gm_ctx *c, const double *x, double *resid, double *val, float *val32,
                      int resid_only) {
  FillArgs a;
  a.resid_only = resid_only;
  a.coor = c->d_coor;
  a.conn = c->d_conn;
  a.fu = c->d_fu;
  a.centroid = c->d_centroid;
  a.tables = c->d_tables;
  a.x = x;
  a.x_old = c->tr_x_old;
  a.xdot_old = c->tr_xdot_old;
  a.cmass = c->tr_cmass;
  a.cold = c->tr_cold;
  a.qs_ptr = c->qs_side.empty() ? nullptr : c->d_qs_ptr;
  a.qs_side = c->d_qs_side;
  a.qs_q = c->d_qs_q;
  a.stab = c->d_stab;
  a.num_nodes = c->num_nodes;
  a.tau_pspg = c->phys.pspg ? gm_pspg_tau(c) : 0.0;
  a.supg_e = c->energy ? c->phys.energy_supg : 0.0;
  a.E = c->lay.total;
  a.off_mp = c->lay.off_mp;
  a.off_cv = c->lay.off_cv;
  a.off_cp = c->lay.off_cp;
  const gm_physics &p = c->phys;
  a.rho = p.rho;
  a.mu0 = p.mu0;
  a.muinf = p.muinf;
  a.lam = p.lam;
  a.nexp = p.nexp;
  a.aexp = p.aexp;
  a.Cp = p.Cp;
  a.kcond = p.kcond;
  a.hsrc = p.hsrc;
  for (int k = 0; k < 3; k++) a.g[k] = p.g[k];
  a.beta = p.beta;
  a.Tref = p.Tref;
  *c->h_flag = 0;  // nothing that could set it is in flight: every call waits for its kernels
  a.flag = c->h_flag;
  int rc = resid_only ? GM_OK : gm_mg_kel_alloc(c);
  if (rc || (rc = elem_buffers(c, !resid_only && c->energy && a.tau_pspg != 0.0))) return rc;
  a.kel = c->d_kel;
  a.re = c->d_re;
  a.ct = c->d_ct;
  if ((rc = assemble(c, a, resid, val, val32))) return rc;
  GM_HIP(hipGetLastError());
  GM_HIP(hipStreamSynchronize(c->stream));
  if (*(volatile int *)c->h_flag) {
    gm_set_error("zero or negative element Jacobian determinant");
    return GM_ERR_ELEM;
  }
  return GM_OK;
}
