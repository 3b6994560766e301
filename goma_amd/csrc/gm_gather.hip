// Element matrices -> MSR matrix, a thread per pair of coupled nodes and row.
//
// The node graph's pairs (row node n, column node m, in the graph's order) are
// the blocks of the matrix: pair p holds the MSR offset of m's first column in
// the rows of n and the list of elements that contain both nodes, each with
// the pair's local position.  A thread sums its row of the pair's block over that
// list, in element order, and writes it once: no colours, no zeroing, no
// read-modify-write, and the same bits every time.  Neighbouring threads write
// neighbouring columns of the same rows.
//
// It is the second half of the assembly (gm_fill.hip) and the scatter of the
// Galerkin coarse levels (gm_mg.hip).
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

// n values at val[pos ..], stored or added.  Stores go out 16 bytes at a time
// (aligned to the value only).
template <int n, typename JT>
__device__ inline void put(JT *val, long long pos, const double *v, bool assign) {
  constexpr int W = 16 / sizeof(JT), M = n / W * W;
  if (!assign) {
#pragma unroll
    for (int k = 0; k < n; k++) val[pos + k] += (JT)v[k];
    return;
  }
  typedef JT Wide __attribute__((ext_vector_type(W), aligned(sizeof(JT))));
#pragma unroll
  for (int k = 0; k < M; k += W) {
    Wide w;
#pragma unroll
    for (int l = 0; l < W; l++) w[l] = (JT)v[k + l];
    *(Wide *)(val + pos + k) = w;
  }
#pragma unroll
  for (int k = M; k < n; k++) val[pos + k] = (JT)v[k];
}

// columns fm .. fm + n - 1 of a row, whose place among the off-diagonals is
// base; the diagonal stands apart and those after it one place earlier
template <int n, typename JT>
__device__ inline void put_row(JT *val, int row, long long base, int fm, const double *v, bool dir, double unit,
                               bool assign) {
  double w[n];
#pragma unroll
  for (int k = 0; k < n; k++) w[k] = dir ? 0.0 : v[k];
  if (row < fm || row >= fm + n) {
    if (assign || !dir) put<n>(val, base - (fm > row ? 1 : 0), w, assign);
    return;
  }
#pragma unroll
  for (int k = 0; k < n; k++) {
    const int col = fm + k;
    if (row == col) {
      const double d = dir ? unit : w[k];
      put<1>(val, row, &d, assign);
    } else if (assign || !dir) {
      put<1>(val, base + k - (col > row ? 1 : 0), &w[k], assign);
    }
  }
}

// A Dirichlet row keeps the unit diagonal of each element at its node
// (put_dirichlet_in_matrix per element, src/bc_dirich.c:44-153); its residual
// is that many times x - V.
//
// Bound by memory: every element-matrix entry read once (8 bytes) and every
// nonzero written once.  Wave a of a workgroup takes row a of the block's 64
// pairs (and the continuity rows a, a + NV, ..): with a thread for all the
// rows of its pair there are a quarter of the waves, and those of the corner
// nodes, eight dependent sources long, are waited for (11^3 elements with
// energy, FP32: 70 us against 86; 16 x 16 QUAD9: 5.9 against 8.0).  The row's
// columns of a pair stand together in the element matrices, two 16-byte reads
// instead of a line for each: 16^3 with energy, FP64, 246 us against 300, 11^3
// FP32 60 against 70.  Pairs in ranges per XCD: two workgroups that share a
// row's lines share an L2 (453 MB read there, 403 of them element matrices);
// most pairs have one source, so the loop is left rolled: 230 and 52 us (3.4
// TB/s).  Two or four pairs a thread (254, 334 us) and half a pair (273) are
// slower.
template <int DIM, int EN, typename JT>
__global__ __launch_bounds__(64 * (DIM + EN)) void k_gather(GatherArgs A, JT *__restrict__ val) {
  constexpr int NVE = DIM == 2 ? 9 : 27, NP = DIM + 1, NV = DIM + EN, NVE2 = NVE * NVE, NT = 64 * NV;
  constexpr int CL = DIM == 2 ? 8 : 20;
  const int blk = xcd_block();
  if (blk >= A.nb_pairs) {
    const int u = (blk - A.nb_pairs) * NT + threadIdx.x;
    if (u >= A.N) return;
    const int k0 = A.gptr[u], k1 = A.gptr[u + 1];
    double s = 0.0;
    if (A.dbc[u]) s = (k1 - k0) * (A.x[u] - A.dbc_val[u]);
    else
      for (int k = k0; k < k1; k++) s += A.re[A.gent[k]];
    A.resid[u] += s;
    return;
  }
  const int a = threadIdx.x >> 6, p = blk * 64 + (threadIdx.x & 63);
  if (p == 0 && a == 0 && A.assign) val[A.N] = (JT)0;  // the unused entry between diagonal and rows
  if (p >= A.npairs) return;
  const int4 P = A.pair[p];
  const int s0 = P.w, s1 = A.pair[p + 1].w, fn = P.x, fm = P.y, ra = P.z & (HAS_P_ROW - 1);
  const bool pc = P.z & HAS_P_COL, pr = P.z & HAS_P_ROW, as = A.assign != 0;
  typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
  {
    const int row = fn + a;
    const bool dir = A.dbc[row] != 0;
    const long long base = (long long)A.bindx[row] + (a < DIM ? ra : A.rank_t[p]);
    double acc[NV + NP];
#pragma unroll
    for (int b = 0; b < NV + NP; b++) acc[b] = 0.0;
    if (!dir)
#pragma unroll 1
      for (int s = s0; s < s1; s++) {
        const int sv = A.src[s], e = sv / NVE2, t = sv - e * NVE2;
        const double *__restrict__ K = A.kel + (size_t)e * A.E, *__restrict__ B = K + (a * NVE2 + t) * NV;
#pragma unroll
        for (int b = 0; b < NV / 2 * 2; b += 2) {
          const Two w = *(const Two *)(B + b);
          acc[b] += w[0];
          acc[b + 1] += w[1];
        }
        if constexpr (NV & 1) acc[NV - 1] += B[NV - 1];
        if (pc && a < DIM && t % NVE == CL) {
          const double *__restrict__ Q = K + A.off_mp + (a * NVE + t / NVE) * NP;
#pragma unroll
          for (int k = 0; k < NP; k++) acc[NV + k] += Q[k];
        }
      }
    if (pc && a < DIM) put_row<NV + NP>(val, row, base, fm, acc, dir, (double)(s1 - s0), as);
    else put_row<NV>(val, row, base, fm, acc, dir, (double)(s1 - s0), as);
  }
  if (!pr) return;
  // continuity rows: velocities, temperature (PSPG only), pressures
#pragma unroll 1
  for (int k = a; k < NP; k += NV) {
    const int row = fn + NV + k;
    const bool dir = A.dbc[row] != 0;
    double acc[NV + NP], nd = 0.0;
#pragma unroll
    for (int b = 0; b < NV + NP; b++) acc[b] = 0.0;
    for (int s = s0; s < s1; s++) {
      const int sv = A.src[s], e = sv / NVE2, t = sv - e * NVE2, i = t / NVE, j = t - i * NVE;
      if (i != CL) continue;
      nd += 1.0;
      const double *__restrict__ K = A.kel + (size_t)e * A.E;
#pragma unroll
      for (int b = 0; b < DIM; b++) acc[b] += K[A.off_cv + (b * NP + k) * NVE + j];
      if (EN && A.ct) acc[NV - 1] += A.ct[(size_t)e * NP * NVE + k * NVE + j];
      if (j == CL)
#pragma unroll
        for (int b = 0; b < NP; b++) acc[NV + b] += K[A.off_cp + k * NP + b];
    }
    const long long base = (long long)A.bindx[row] + ra;
    if (pc) put_row<NV + NP>(val, row, base, fm, acc, dir, nd, as);
    else put_row<NV>(val, row, base, fm, acc, dir, nd, as);
  }
}

// The pairs' descriptions, one thread per row node: pair p's sources are the
// (k, l) places of its two nodes in a common element, element by element; the
// pairs of node n hold nve of them for each of its places.
__global__ __launch_bounds__(256) void k_pairs(int nn, int nve, int nv, const int *__restrict__ fu,
                                               const int *__restrict__ nn_ptr, const int *__restrict__ nn_list,
                                               const int *__restrict__ eptr, const int *__restrict__ elist,
                                               int4 *__restrict__ pair, int *__restrict__ rank_t,
                                               int *__restrict__ src) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n > nn) return;
  if (n == nn) {
    pair[nn_ptr[nn]] = make_int4(0, 0, 0, eptr[nn] * nve);
    return;
  }
  const int k0 = eptr[n], k1 = eptr[n + 1], fn = fu[n], pr = fu[n + 1] - fn > nv ? HAS_P_ROW : 0;
  int ra = 0, rt = 0, at = k0 * nve;
  for (int p = nn_ptr[n]; p < nn_ptr[n + 1]; p++) {
    const int m = nn_list[p], l = fu[m + 1] - fu[m];
    pair[p] = make_int4(fn, fu[m], ra | (l > nv ? HAS_P_COL : 0) | pr, at);
    rank_t[p] = rt;
    ra += l;
    rt += min(l, nv);
    for (int k = k0; k < k1; k++) {
      const int e = elist[k] / nve, i = elist[k] - e * nve;
      for (int q = eptr[m]; q < eptr[m + 1]; q++)
        if (elist[q] / nve == e) src[at++] = e * nve * nve + i * nve + elist[q] - e * nve;
    }
  }
}

}  // namespace

// The pairs' descriptions from the node graph and the connectivity, and each
// unknown's places in the element vectors (d_mg_gptr / d_mg_gent, shared with
// the additive smoother).
int gm_gather_setup(gm_ctx *c) {
  if (c->d_pair) return GM_OK;
  const int nn = c->num_nodes, ne = c->num_elems, nve = c->nve;
  const size_t npairs = c->nn_list.size(), places = (size_t)ne * nve;
  // (the 32-bit row pointers of the matrix end far below this)
  if (places * nve >= (1ull << 31) || npairs >= (1ull << 31) - 512) {
    gm_set_error("too many elements for the assembly's pair lists (%d)", ne);
    return GM_ERR_ARG;
  }
  std::vector<int> eptr(nn + 1, 0), elist(places);
  for (size_t k = 0; k < places; k++) eptr[c->conn[k] + 1]++;
  for (int n = 0; n < nn; n++) eptr[n + 1] += eptr[n];
  {
    std::vector<int> at(eptr.begin(), eptr.end() - 1);
    for (size_t k = 0; k < places; k++) elist[at[c->conn[k]]++] = (int)k;
  }
  int *d_eptr = nullptr, *d_elist = nullptr;
  int4 *pair = nullptr;
  auto build = [&]() -> int {
    int rc;
    if ((rc = up(&d_eptr, eptr)) || (rc = up(&d_elist, elist)) || (rc = gm_unknown_places(c))) return rc;
    GM_HIP(hipMalloc(&pair, (npairs + 1) * sizeof(int4)));
    if (!c->d_rank_t) GM_HIP(hipMalloc(&c->d_rank_t, std::max<size_t>(npairs, 1) * sizeof(int)));
    if (!c->d_src) GM_HIP(hipMalloc(&c->d_src, places * nve * sizeof(int)));
    k_pairs<<<nn / 256 + 1, 256, 0, c->stream>>>(nn, nve, c->nv, c->d_fu, c->d_nn_ptr, c->d_nn_list, d_eptr, d_elist,
                                                 pair, c->d_rank_t, c->d_src);
    GM_HIP(hipGetLastError());
    GM_HIP(hipStreamSynchronize(c->stream));
    return GM_OK;
  };
  const int rc = build();
  (void)hipFree(d_eptr);
  (void)hipFree(d_elist);
  if (rc) (void)hipFree(pair);
  else c->d_pair = pair;
  return rc;
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
  const int nt = 64 * c->nv;
  A.nb_pairs = (A.npairs + 63) / 64;
  const int blocks = A.nb_pairs + (re ? (c->N + nt - 1) / nt : 0);
  if (!blocks) return GM_OK;
  const double nnz = (double)c->nval - 1.0, vs = val32 ? 4.0 : 8.0;
  const double bytes = (mat ? (double)c->num_elems * c->lay.total * 8.0 + nnz * vs * (assign ? 1.0 : 2.0) +
                                  20.0 * A.npairs + 4.0 * c->num_elems * c->nve * c->nve
                            : 0.0) +
                       (re ? (double)c->num_elems * (c->nv * c->nve + c->np) * 12.0 + 20.0 * c->N : 0.0);
  auto go = [&](auto kern, auto *v) { gm_launch(prof, id, bytes, kern, dim3(blocks), dim3(nt), 0, s, A, v); };
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
