// Element matrices -> MSR matrix, one thread per pair of coupled nodes.
//
// The node graph's pairs (row node n, column node m, in the graph's order) are
// the blocks of the matrix: pair p holds the MSR offset of m's first column in
// the rows of n and the list of elements that contain both nodes, each with
// the pair's local position.  A thread sums its pair's block over that list,
// in element order, and writes it once: no colours, no zeroing, no
// read-modify-write, and the same bits every time.  Neighbouring threads write
// neighbouring columns of the same rows.
//
// It is the second half of the QUAD9 assembly (gm_fill.hip) and the scatter
// of the Galerkin coarse levels (gm_mg.hip).
#include <algorithm>
#include <vector>

#include "gm_launch.h"

namespace {

template <typename T>
int up(T **d, const std::vector<T> &h) {
  GM_HIP(hipMalloc(d, std::max<size_t>(h.size(), 1) * sizeof(T)));
  if (!h.empty()) GM_HIP(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  return GM_OK;
}

struct GatherArgs {
  const int4 *pair;   // (first unknown of n, of m, MSR offset | flags, first source)
  const int *rank_t;  // offset in the energy rows, which have no pressure columns
  const int *src;     // element * nve^2 + i * nve + j
  const double *kel, *ct;
  const int *bindx;
  const signed char *dbc;
  long long E, off_mp, off_cv, off_cp;
  int npairs, N, assign;
  // residual rows (re null: none): x_u of a Dirichlet row counts once per element
  const int *gptr, *gent;
  const double *re, *x, *dbc_val;
  double *resid;
  int nb_pairs;  // blocks of the matrix; the rest sum the residual
};

constexpr int HAS_P_COL = 1 << 30;  // m carries pressure unknowns
constexpr int HAS_P_ROW = 1 << 29;  // n does

template <typename JT>
__device__ inline void put(JT *val, long long pos, double v, bool assign) {
  if (assign) val[pos] = (JT)v;
  else val[pos] += (JT)v;
}

// A Dirichlet row keeps the unit diagonal of each element at its node
// (put_dirichlet_in_matrix per element, src/bc_dirich.c:44-153); its residual
// is that many times x - V.
//
// Bound by memory: every element-matrix entry read once (8 bytes) and every
// nonzero written once.  A thread takes its pair through all the rows of n,
// so the pair's description is read once and its loads are independent.
template <int DIM, int EN, typename JT>
__global__ __launch_bounds__(256) void k_gather(GatherArgs A, JT *__restrict__ val) {
  constexpr int NVE = DIM == 2 ? 9 : 27, NP = DIM + 1, NV = DIM + EN, NVE2 = NVE * NVE;
  constexpr int CL = DIM == 2 ? 8 : 20;
  if ((int)blockIdx.x >= A.nb_pairs) {
    const int u = ((int)blockIdx.x - A.nb_pairs) * 256 + threadIdx.x;
    if (u >= A.N) return;
    const int k0 = A.gptr[u], k1 = A.gptr[u + 1];
    double s = 0.0;
    if (A.dbc[u]) s = (k1 - k0) * (A.x[u] - A.dbc_val[u]);
    else
      for (int k = k0; k < k1; k++) s += A.re[A.gent[k]];
    A.resid[u] += s;
    return;
  }
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p == 0 && A.assign) val[A.N] = (JT)0;  // the unused entry between diagonal and rows
  if (p >= A.npairs) return;
  const int4 P = A.pair[p];
  const int s0 = P.w, s1 = A.pair[p + 1].w, fn = P.x, fm = P.y, ra = P.z & (HAS_P_ROW - 1);
  const int rt = EN ? A.rank_t[p] : 0;
  const bool pc = P.z & HAS_P_COL, pr = P.z & HAS_P_ROW, as = A.assign != 0;
  double acc[NV][NV], accp[DIM][NP];
#pragma unroll
  for (int a = 0; a < NV; a++)
#pragma unroll
    for (int b = 0; b < NV; b++) acc[a][b] = 0.0;
#pragma unroll
  for (int a = 0; a < DIM; a++)
#pragma unroll
    for (int k = 0; k < NP; k++) accp[a][k] = 0.0;
  for (int s = s0; s < s1; s++) {
    const int sv = A.src[s], e = sv / NVE2, t = sv - e * NVE2;
    const double *__restrict__ K = A.kel + (size_t)e * A.E;
#pragma unroll
    for (int a = 0; a < NV; a++)
#pragma unroll
      for (int b = 0; b < NV; b++) acc[a][b] += K[(a * NV + b) * NVE2 + t];
    if (pc && t % NVE == CL) {
      const double *__restrict__ Q = K + A.off_mp + (t / NVE) * NP;
#pragma unroll
      for (int a = 0; a < DIM; a++)
#pragma unroll
        for (int k = 0; k < NP; k++) accp[a][k] += Q[a * NVE * NP + k];
    }
  }
#pragma unroll
  for (int a = 0; a < NV; a++) {
    const int row = fn + a;
    const bool dir = A.dbc[row] != 0;
    const long long base = (long long)A.bindx[row] + (a < DIM ? ra : rt) - (fm > row ? 1 : 0);
#pragma unroll
    for (int b = 0; b < NV; b++) {
      const int col = fm + b;
      const bool diag = row == col;
      if (dir && !diag && !as) continue;
      const double v = dir ? (diag ? (double)(s1 - s0) : 0.0) : acc[a][b];
      // the columns of m after the row's own unknown stand one place earlier
      const long long pos = diag ? row : base + b - (fm <= row && col > row ? 1 : 0);
      put(val, pos, v, as);
    }
    if (pc && a < DIM) {
#pragma unroll
      for (int k = 0; k < NP; k++) {
        if (dir && !as) continue;
        put(val, base + NV + k - (fm <= row && fm + NV + k > row ? 1 : 0), dir ? 0.0 : accp[a < DIM ? a : 0][k], as);
      }
    }
  }
  if (!pr) return;
  // continuity rows: velocities, temperature (PSPG only), pressures
#pragma unroll 1
  for (int k = 0; k < NP; k++) {
    const int row = fn + NV + k;
    const bool dir = A.dbc[row] != 0;
    double c[NV], q[NP], nd = 0.0;
#pragma unroll
    for (int b = 0; b < NV; b++) c[b] = 0.0;
#pragma unroll
    for (int b = 0; b < NP; b++) q[b] = 0.0;
    for (int s = s0; s < s1; s++) {
      const int sv = A.src[s], e = sv / NVE2, t = sv - e * NVE2, i = t / NVE, j = t - i * NVE;
      if (i != CL) continue;
      nd += 1.0;
      const double *__restrict__ K = A.kel + (size_t)e * A.E;
#pragma unroll
      for (int b = 0; b < DIM; b++) c[b] += K[A.off_cv + (b * NP + k) * NVE + j];
      if (EN && A.ct) c[NV - 1] += A.ct[(size_t)e * NP * NVE + k * NVE + j];
      if (j == CL)
#pragma unroll
        for (int b = 0; b < NP; b++) q[b] += K[A.off_cp + k * NP + b];
    }
    const long long base = (long long)A.bindx[row] + ra - (fm > row ? 1 : 0);
#pragma unroll
    for (int b = 0; b < NV + NP; b++) {
      if (b >= NV && !pc) continue;
      const int col = fm + b;
      const bool diag = row == col;
      if (dir && !diag && !as) continue;
      const double v = dir ? (diag ? nd : 0.0) : (b < NV ? c[b < NV ? b : 0] : q[b >= NV ? b - NV : 0]);
      const long long pos = diag ? row : base + b - (fm <= row && col > row ? 1 : 0);
      put(val, pos, v, as);
    }
  }
}

}  // namespace

// The pairs' descriptions from the node graph and the connectivity, and each
// unknown's places in the element vectors (d_mg_gptr / d_mg_gent, shared with
// the additive smoother).
int gm_gather_setup(gm_ctx *c) {
  if (c->d_pair) return GM_OK;
  const int nn = c->num_nodes, ne = c->num_elems, nve = c->nve, nve2 = nve * nve, nv = c->nv, np = c->np;
  const size_t npairs = c->nn_list.size();
  if ((long long)ne * nve2 >= (1LL << 31) || npairs >= (1ull << 31) - 512) {
    gm_set_error("too many elements for the assembly's pair lists (%d)", ne);
    return GM_ERR_ARG;
  }
  std::vector<int> eptr(nn + 1, 0), elist((size_t)ne * nve);
  for (size_t k = 0; k < (size_t)ne * nve; k++) eptr[c->conn[k] + 1]++;
  for (int n = 0; n < nn; n++) eptr[n + 1] += eptr[n];
  {
    std::vector<int> fp(eptr.begin(), eptr.end() - 1);
    for (int e = 0; e < ne; e++)
      for (int i = 0; i < nve; i++) elist[fp[c->conn[(size_t)e * nve + i]]++] = e * nve + i;
  }
  std::vector<int4> pair(npairs + 1);
  std::vector<int> rank_t(npairs), cnt(npairs, 0);
  auto find = [&](int n, int m) {
    return (size_t)(std::lower_bound(c->nn_list.begin() + c->nn_ptr[n], c->nn_list.begin() + c->nn_ptr[n + 1], m) -
                    c->nn_list.begin());
  };
  auto len = [&](int n) { return c->first_unknown[n + 1] - c->first_unknown[n]; };
#pragma omp parallel for schedule(dynamic, 1024)
  for (int n = 0; n < nn; n++) {
    int ra = 0, rt = 0;
    for (int p = c->nn_ptr[n]; p < c->nn_ptr[n + 1]; p++) {
      const int m = c->nn_list[p], l = len(m);
      pair[p] = make_int4(c->first_unknown[n], c->first_unknown[m],
                          ra | (l > nv ? HAS_P_COL : 0) | (len(n) > nv ? HAS_P_ROW : 0), 0);
      rank_t[p] = rt;
      ra += l;
      rt += std::min(l, nv);
    }
    for (int k = eptr[n]; k < eptr[n + 1]; k++)
      for (int j = 0; j < nve; j++) cnt[find(n, c->conn[(size_t)(elist[k] / nve) * nve + j])]++;
  }
  int total = 0;
  for (size_t p = 0; p < npairs; p++) {
    pair[p].w = total;
    total += cnt[p];
  }
  pair[npairs] = make_int4(0, 0, 0, total);
  std::vector<int> src(total);
#pragma omp parallel for schedule(dynamic, 1024)
  for (int n = 0; n < nn; n++) {
    for (int p = c->nn_ptr[n]; p < c->nn_ptr[n + 1]; p++) cnt[p] = pair[p].w;
    for (int k = eptr[n]; k < eptr[n + 1]; k++) {
      const int e = elist[k] / nve, i = elist[k] - e * nve;
      for (int j = 0; j < nve; j++) src[cnt[find(n, c->conn[(size_t)e * nve + j])]++] = e * nve2 + i * nve + j;
    }
  }
  int rc;
  if ((rc = up(&c->d_src, src)) || (rc = up(&c->d_rank_t, rank_t)) || (rc = gm_unknown_places(c)) ||
      (rc = up(&c->d_pair, pair)))
    return rc;
  return GM_OK;
}

// Local dof li of element e (nodal variables node-blocked by variable, then
// the element's P1 dofs) is unknown g: gptr[g] .. gptr[g + 1] list its places
// e * nl + li, element by element.
int gm_unknown_places(gm_ctx *c) {
  if (c->d_mg_gptr) return GM_OK;
  const int nl = c->nv * c->nve + c->np;
  std::vector<int> gptr(c->N + 1, 0), gent((size_t)c->num_elems * nl);
  auto dof = [&](int e, int li) {
    if (li < c->nv * c->nve) {
      const int a = li / c->nve, i = li - a * c->nve;
      return c->first_unknown[c->conn[(size_t)e * c->nve + i]] + a;
    }
    return c->first_unknown[c->elem_centroid[e]] + c->dim + c->energy + (li - c->nv * c->nve);
  };
  for (int e = 0; e < c->num_elems; e++)
    for (int li = 0; li < nl; li++) gptr[dof(e, li) + 1]++;
  for (int u = 0; u < c->N; u++) gptr[u + 1] += gptr[u];
  std::vector<int> fill(gptr.begin(), gptr.end() - 1);
  for (int e = 0; e < c->num_elems; e++)
    for (int li = 0; li < nl; li++) gent[fill[dof(e, li)]++] = e * nl + li;
  int rc = up(&c->d_mg_gent, gent);
  return rc ? rc : up(&c->d_mg_gptr, gptr);
}

// val (FP64) or val32 from the element matrices kel of context c, on stream s,
// stored (assign) or added; with re, also resid += the element residuals (only
// those when val and val32 are null).  ct: continuity x temperature entries
// [elem][np][nve], or null.
int gm_gather(gm_ctx *prof, int id, gm_ctx *c, hipStream_t s, const double *kel, const double *ct, double *val,
              float *val32, int assign, const double *re, const double *x, double *resid) {
  GatherArgs A;
  A.pair = c->d_pair;
  A.rank_t = c->d_rank_t;
  A.src = c->d_src;
  A.kel = kel;
  A.ct = ct;
  A.bindx = c->d_bindx;
  A.dbc = c->d_dbc;
  A.E = c->lay.total;
  A.off_mp = c->lay.off_mp;
  A.off_cv = c->lay.off_cv;
  A.off_cp = c->lay.off_cp;
  A.N = c->N;
  A.assign = assign;
  A.gptr = c->d_mg_gptr;
  A.gent = c->d_mg_gent;
  A.re = re;
  A.x = x;
  A.dbc_val = c->d_dbc_val;
  A.resid = resid;
  const bool mat = val || val32;
  A.npairs = mat ? (int)c->nn_list.size() : 0;
  A.nb_pairs = (A.npairs + 255) / 256;
  const int blocks = A.nb_pairs + (re ? (c->N + 255) / 256 : 0);
  if (!blocks) return GM_OK;
  const double nnz = (double)c->nval - 1.0, vs = val32 ? 4.0 : 8.0;
  const double bytes = (mat ? (double)c->num_elems * c->lay.total * 8.0 + nnz * vs * (assign ? 1.0 : 2.0) +
                                  20.0 * A.npairs + 4.0 * c->num_elems * c->nve * c->nve
                            : 0.0) +
                       (re ? (double)c->num_elems * (c->nv * c->nve + c->np) * 12.0 + 20.0 * c->N : 0.0);
  auto go = [&](auto kern, auto *v) { gm_launch(prof, id, bytes, kern, dim3(blocks), dim3(256), 0, s, A, v); };
  if (val32) {
    if (c->dim == 2) go(c->energy ? k_gather<2, 1, float> : k_gather<2, 0, float>, val32);
    else go(c->energy ? k_gather<3, 1, float> : k_gather<3, 0, float>, val32);
  } else {
    if (c->dim == 2) go(c->energy ? k_gather<2, 1, double> : k_gather<2, 0, double>, val);
    else go(c->energy ? k_gather<3, 1, double> : k_gather<3, 0, double>, val);
  }
  GM_HIP(hipGetLastError());
  return GM_OK;
}
