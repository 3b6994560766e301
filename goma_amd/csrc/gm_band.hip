// Banded LU factorisation and solve of the row-sum-scaled Jacobian, without
// pivoting, in Goma's unknown order: a direct solver on the GPU for the
// Newton systems where iterative preconditioners stall -- the role of Goma's
// direct solvers (Solution Algorithm = lu, Goma's default, src/mm_input.c:5904;
// umf / lu dispatch in src/mm_sol_nonlinear.c:1624-1681) -- behind the same
// GMRES interface as the other preconditioners.
//
// Storage.  With kl / ku the lower / upper bandwidths of the MSR graph, the
// band lives column-major in ld = kl + ku + 1 + 2 MG entries per column,
// A(i, j) at ab[off + i + j * lda] with off = MG + ku and lda = ld - 1, for
// j - ku - MG <= i <= j + kl + MG.  The MG-entry margins above and below the
// band let every panel step treat its window as a plain dense matrix: window
// entries outside the band start at zero and stay exactly zero (each of their
// updates has a zero factor).  Without pivoting no fill leaves the band.
//
// Factorisation, right-looking in panels of NB = 64 columns, with the inverse
// triangles of each diagonal block, so that everything but that block is a
// matrix product (FP64 matrix cores):
//   k_band_diag    A11 = L11 U11, as L11^-1 and U11^-1, of the first panel;
//                  later ones come at the end of the previous update, from the
//                  workgroup whose tile holds them;
//   k_band_panel   L21 = A21 U11^-1 and U12 = L11^-1 A12, a 64 x 64 tile each;
//   k_band_update  A22 -= L21 U12 by 64 x 64 tiles.
// The chain of panels bounds it for bandwidths of a few thousand, and in it
// the diagonal block.
// Solve: forward and backward by pairs of panels (SB = 128 unknowns), whose
// operators k_band_ops forms for all pairs at once after the factorisation;
// one launch per pair and direction.  Zero pivots are reported
// (GM_ERR_PIVOT), never divided by.
// Where a diagonal block's triangles are ill-conditioned (saddle points),
// products with their inverses leave more than triangular substitution does, so
// an FP64 solve is refined once against the matrix.  Relative residual of one
// solve, geometric means of six states, substitution / inverses / inverses
// refined: 8 x 8 shear-thinning 5.6e-12 / 2.5e-11 / 4.2e-14, 3^3 cavity
// 1.4e-12 / 1.6e-11 (one state 1000 times the substitution's) / 1.9e-15, 32 x 32
// shear-thinning 6.7e-13 / 6.2e-13 / 5.1e-14.  Newton on the 40 x 40
// shear-thinning case: 690 / 204 / 250 ms.
#include <algorithm>
#include <cmath>
#include <vector>

#include "gm_launch.h"

namespace {

constexpr int NB = 64;  // panel width
constexpr int MG = NB;  // storage margin above and below the band

template <typename T>
__global__ __launch_bounds__(256) void k_band_zero(size_t n, T *__restrict__ p) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = T(0);
}

template <typename VT, typename T>
__global__ __launch_bounds__(256) void k_band_load(int N, const VT *__restrict__ val,
                                                   const int *__restrict__ bindx, T *__restrict__ ab,
                                                   long long off, long long lda) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  ab[off + i + (size_t)i * lda] = (T)val[i];
  for (int k = bindx[i]; k < bindx[i + 1]; k++) ab[off + i + (size_t)bindx[k] * lda] = (T)val[k];
}

constexpr int SB = 2 * NB;  // unknowns a solve step takes
constexpr int LDT = NB + 2; // LDS row of a 64 x 64 block
constexpr int OPS = SB * SB * 2;  // operators of one pair of panels
constexpr int TRI = 2 * NB * NB;   // inverse triangles of one panel

typedef double d4v __attribute__((ext_vector_type(4)));

// D[m][n] = sum_k fa(k, m) fb(k, n) over k < 64 on one wave's 32 x 32 quadrant
// (m0, n0) of a 64 x 64 block; the lane holds rows m0 + 16 u + l / 16 + 4 r and
// column n0 + 16 v + l % 16 (v_mfma_f64_16x16x4f64).
template <typename FA, typename FB>
__device__ __forceinline__ void product64(int m0, int n0, FA fa, FB fb, d4v (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, kk = lane >> 4;
#pragma unroll
  for (int k0 = 0; k0 < NB; k0 += 16) {
    double a[4][2], b[4][2];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 2; u++) {
        a[q][u] = fa(k0 + 4 * q + kk, m0 + 16 * u + r16);
        b[q][u] = fb(k0 + 4 * q + kk, n0 + 16 * u + r16);
      }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
          acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q][u], b[q][v], acc[u][v], 0, 0, 0);
  }
}
__device__ inline void clear(d4v (&acc)[2][2]) {
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++) acc[u][v] = d4v{0.0, 0.0, 0.0, 0.0};
}
// f(row, column, value) over the quadrant's entries that this lane holds
template <typename F>
__device__ inline void each(int m0, int n0, const d4v (&acc)[2][2], F f) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int r = 0; r < 4; r++) f(m0 + 16 * u + (lane >> 4) + 4 * r, n0 + 16 * v + (lane & 15), acc[u][v][r]);
}

// LU (no pivoting) of the 64 x 64 block s (LDS, overwritten) by all 256
// threads, as the inverse triangles L^-1 (column-major, tri) and U^-1
// (row-major, tri + 64 x 64), each as its panel product reads it.  Both
// inverses grow in place, by blocks of 16: step K inverts the triangles of its
// diagonal block, L_KK^-1 and U_KK^-1; multiplies its block row by the one
// (left of K: L^-1; right: U) and its block column by the other (above: U^-1;
// below: L); then the products of the two are subtracted below K and, right of
// K, above it, and the row's and the column's other halves start as
// -U_KK^-1 U_Kj and -L_iK L_KK^-1.  The block products run on the matrix cores.
// A diagonal block is a row per lane of one wave, its 16 steps a chain of DPP
// broadcasts without LDS or barriers: 0.11 us a step, 16 us for the block, where
// steps through LDS with a barrier each took 0.41 (a panel's launch 33.6 us,
// 28.8 now).
__device__ __forceinline__ void block_triangles(double (*s)[LDT], double *__restrict__ tri, int *flag) {
  constexpr int B = 16, LB = B + 1;
  // block column and row of step K, the diagonal block's inverse triangles
  __shared__ double s_f[4][B][LB], s_g[4][B][LB], s_tl[B][LB], s_tu[B][LB];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  // two block products at a time: D[lq + 4 r][l16] = sum_k a[l16][k] b[k][l16]
  auto products = [&](const double *a0, int la0, const double *b0, int lb0, const double *a1, int la1, const double *b1,
                      int lb1, d4v &D0, d4v &D1) {
    double x[2][4], y[2][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int k = 4 * q + lq;
      x[0][q] = a0[l16 * la0 + k];
      y[0][q] = b0[k * lb0 + l16];
      x[1][q] = a1[l16 * la1 + k];
      y[1][q] = b1[k * lb1 + l16];
    }
    D0 = D1 = d4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; q++) {
      D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[0][q], y[0][q], D0, 0, 0, 0);
      D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[1][q], y[1][q], D1, 0, 0, 0);
    }
  };
#pragma unroll 1
  for (int K = 0; K < 4; K++) {
    const int k0 = B * K;
    if (wave == 0) {
      // every DPP row holds the block, a row per lane; a row's right part waits
      // for its scale until the end
      double P[B], scale = 0.0;
      bool zero = false;
#pragma unroll
      for (int j = 0; j < B; j++) P[j] = s[k0 + l16][k0 + j];
#pragma unroll
      for (int k = 0; k < B; k++) {
        double piv = row_bcast(P[k], k);
        if (piv == 0.0) {
          zero = true;
          piv = 1.0;
        }
        const double d = reciprocal(piv);
        const bool is = l16 == k, below = l16 > k;
        const double f = is ? 0.0 : P[k] * d, g = below ? f : 0.0;
        scale = is ? -d : scale;
#pragma unroll
        for (int j = k + 1; j < B; j++) P[j] = fma(row_bcast(P[j], k), -f, P[j]);
#pragma unroll
        for (int j = 0; j < k; j++) P[j] = fma(row_bcast(P[j], k), -g, P[j]);
        P[k] = is ? -1.0 : below ? -f : f;
      }
      // a DPP row stores a quarter of the columns
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int j = 4 * lq + c;
        const double w = lq < 2 ? (lq == 0 ? P[c] : P[4 + c]) : (lq == 2 ? P[8 + c] : P[12 + c]);
        s_tl[l16][j] = j < l16 ? w : j == l16 ? 1.0 : 0.0;
        s_tu[l16][j] = j >= l16 ? w * scale : 0.0;
      }
      if (zero && lane == 0) atomicOr(flag, 1);
    }
    __syncthreads();
    if (wave < 3) {  // the block row and column
      const int m = wave < K ? wave : wave + 1, m0 = B * m;
      d4v G, F;
      products(&s_tl[0][0], LB, &s[k0][m0], LDT, &s[m0][k0], LDT, &s_tu[0][0], LB, G, F);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = lq + 4 * r;
        s_g[m][i][l16] = G[r];
        s_f[m][i][l16] = F[r];
        if (m < K) {  // final
          s[k0 + i][m0 + l16] = G[r];
          s[m0 + i][k0 + l16] = F[r];
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = lq + 4 * r;
        s[k0 + i][k0 + l16] = i > l16 ? s_tl[i][l16] : s_tu[i][l16];
      }
    }
    __syncthreads();
    // the blocks below K and, right of K, above it; then the two halves of row
    // and column K
    const int nb = 3 - K, nu = 3 * nb + K * nb, nt = nu + 2 * nb;
    auto task = [&](int t, const double *&a, const double *&b, double *&out, bool &sub) {
      sub = t < nu;
      int i = K, j = K;
      if (t < 3 * nb) {
        i = K + 1 + t / 3;
        j = t % 3 < K ? t % 3 : t % 3 + 1;
      } else if (t < nu) {
        i = (t - 3 * nb) / nb;
        j = K + 1 + (t - 3 * nb) % nb;
      } else if (t < nu + nb) {
        i = K + 1 + t - nu;
      } else {
        j = K + 1 + t - nu - nb;
      }
      a = i == K ? &s_tu[0][0] : &s_f[i][0][0];
      b = j == K ? &s_tl[0][0] : &s_g[j][0][0];
      out = &s[B * i][B * j];
    };
    for (int t = wave; t < nt; t += 8) {
      const double *a[2], *b[2];
      double *out[2];
      bool sub[2];
      const bool two = t + 4 < nt;
      task(t, a[0], b[0], out[0], sub[0]);
      task(two ? t + 4 : t, a[1], b[1], out[1], sub[1]);
      d4v D[2];
      products(a[0], LB, b[0], LB, a[1], LB, b[1], LB, D[0], D[1]);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        if (h && !two) break;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          double *o = out[h] + (lq + 4 * r) * LDT + l16;
          *o = (sub[h] ? *o : 0.0) - D[h][r];
        }
      }
    }
    __syncthreads();
  }
#pragma unroll 4
  for (int t = tid; t < NB * NB; t += 256) {
    const int j = t >> 6, i = t & 63;
    const double l = s[i][j], u = s[j][i];
    tri[t] = i > j ? l : i == j ? 1.0 : 0.0;
    tri[NB * NB + t] = j <= i ? u : 0.0;
  }
}

// Inverse triangles of the panel at j0 (kb columns, padded with the identity).
template <typename T>
__global__ __launch_bounds__(256) void k_band_diag(int j0, int kb, const T *__restrict__ ab, long long off,
                                                   long long lda, double *__restrict__ tri, int *flag) {
  __shared__ double s[NB][LDT];
  const T *__restrict__ base = ab + off;
  for (int t = threadIdx.x; t < NB * NB; t += 256) {
    const int j = t >> 6, i = t & 63;
    s[i][j] = (i < kb && j < kb) ? (double)base[(j0 + i) + (size_t)(j0 + j) * lda] : (i == j ? 1.0 : 0.0);
  }
  __syncthreads();
  block_triangles(s, tri, flag);
}

// Workgroups [0, rt): 64 rows of L21 = A21 U11^-1; [rt, gridDim.x): 64 columns
// of U12 = L11^-1 A12; in place, the window's rows [j0 + 64, re) and columns
// [j0 + 64, ce).  The products are formed so that a column's entries of the
// band lie along the lanes.
template <typename T>
__global__ __launch_bounds__(256) void k_band_panel(int j0, int re, int ce, int rt, T *__restrict__ ab,
                                                    long long off, long long lda,
                                                    const double *__restrict__ tri) {
  __shared__ double s_u[NB][LDT];  // A12 [k][column]
  T *__restrict__ base = ab + off;
  const int tid = threadIdx.x, wave = tid >> 6, m0 = (wave >> 1) * 32, n0 = (wave & 1) * 32;
  d4v acc[2][2];
  clear(acc);
  if ((int)blockIdx.x < rt) {
    const int r0 = j0 + NB + blockIdx.x * NB;
    const double *U = tri + NB * NB;
    product64(m0, n0, [&](int k, int m) { return U[k * NB + m]; },
              [&](int k, int i) {
                return r0 + i < re ? (double)base[(size_t)(r0 + i) + (size_t)(j0 + k) * lda] : 0.0;
              },
              acc);
    __syncthreads();  // every wave has read its rows
    each(m0, n0, acc, [&](int m, int i, double v) {
      if (r0 + i < re) base[(size_t)(r0 + i) + (size_t)(j0 + m) * lda] = (T)v;
    });
  } else {
    const int c0 = j0 + NB + ((int)blockIdx.x - rt) * NB;
    for (int t = tid; t < NB * NB; t += 256) {
      const int j = t >> 6, k = t & 63;
      s_u[k][j] = c0 + j < ce ? (double)base[(size_t)(j0 + k) + (size_t)(c0 + j) * lda] : 0.0;
    }
    __syncthreads();
    product64(m0, n0, [&](int k, int j) { return s_u[k][j]; }, [&](int k, int i) { return tri[k * NB + i]; }, acc);
    each(m0, n0, acc, [&](int j, int i, double v) {
      if (c0 + j < ce) base[(size_t)(j0 + i) + (size_t)(c0 + j) * lda] = (T)v;
    });
  }
}

// One 64 x 64 tile of A22 -= L21 U12 for the panel at j0, formed transposed so
// that the band's columns are read and written along their rows.  With next >
// 0, workgroup (0, 0), whose tile holds the next panel's diagonal block, now
// final, takes the inverse triangles of its next x next corner into
// tri_next.  Measured at bandwidth 620 (FP64): 38 us a panel (this
// launch and k_band_panel) against 118 with an LU in LDS, two barriers a
// column, and a thread's triangular solve per row and column.
template <typename T>
__global__ __launch_bounds__(256) void k_band_update(int j0, int re, int ce, int next, T *__restrict__ ab,
                                                     long long off, long long lda,
                                                     double *__restrict__ tri_next, int *flag) {
  __shared__ double s_u[NB][LDT];  // U12 [k][column]; then the updated tile of workgroup (0, 0)
  T *__restrict__ base = ab + off;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m0 = (wave >> 1) * 32, n0 = (wave & 1) * 32;
  const int r0 = j0 + NB + blockIdx.x * NB, c0 = j0 + NB + blockIdx.y * NB;
  for (int t = tid; t < NB * NB; t += 256) {
    const int j = t >> 6, k = t & 63;
    s_u[k][j] = c0 + j < ce ? (double)base[(size_t)(j0 + k) + (size_t)(c0 + j) * lda] : 0.0;
  }
  double cv[2][2][4];  // the tile itself, loaded ahead of the product
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int j = m0 + 16 * u + (lane >> 4) + 4 * r, i = n0 + 16 * v + (lane & 15);
        cv[u][v][r] = (r0 + i < re && c0 + j < ce) ? (double)base[(size_t)(r0 + i) + (size_t)(c0 + j) * lda] : 0.0;
      }
  __syncthreads();
  d4v acc[2][2];
  clear(acc);
  product64(m0, n0, [&](int k, int j) { return s_u[k][j]; },
            [&](int k, int i) {
              return r0 + i < re ? (double)base[(size_t)(r0 + i) + (size_t)(j0 + k) * lda] : 0.0;
            },
            acc);
  const bool fuse = next > 0 && blockIdx.x == 0 && blockIdx.y == 0;
  if (fuse) __syncthreads();  // uniform per workgroup: s_u is reused below
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int j = m0 + 16 * u + (lane >> 4) + 4 * r, i = n0 + 16 * v + (lane & 15);
        const double c = cv[u][v][r] - acc[u][v][r];
        if (r0 + i < re && c0 + j < ce) base[(size_t)(r0 + i) + (size_t)(c0 + j) * lda] = (T)c;
        if (fuse) s_u[i][j] = (i < next && j < next) ? (double)(T)c : (i == j ? 1.0 : 0.0);
      }
  if (!fuse) return;
  __syncthreads();
  block_triangles(s_u, tri_next, flag);
}

// Operators of one pair of panels (0, 1) from their inverse triangles and the
// couplings L10, U01: column-major 128 x 128
//   F = [L0^-1 0; -L1^-1 L10 L0^-1  L1^-1]   (forward:  y = F w)
//   G = [U0^-1 -U0^-1 U01 U1^-1; 0 U1^-1]    (backward: x = G w)
// A missing second panel has the identity and no couplings.
template <typename T>
__global__ __launch_bounds__(256) void k_band_ops(int N, const T *__restrict__ ab, long long off, long long lda,
                                                  int kl, int ku, int npanel,
                                                  const double *__restrict__ tri, double *__restrict__ ops) {
  __shared__ double s_t[NB][LDT];
  const T *__restrict__ base = ab + off;
  const int tid = threadIdx.x, wave = tid >> 6, m0 = (wave >> 1) * 32, n0 = (wave & 1) * 32;
  const int j0 = blockIdx.x * SB, j1 = j0 + NB;
  const bool two = 2 * (int)blockIdx.x + 1 < npanel;
  const double *L0 = tri + (size_t)2 * blockIdx.x * TRI, *U0 = L0 + NB * NB, *L1 = L0 + TRI, *U1 = L1 + NB * NB;
  double *F = ops + (size_t)blockIdx.x * OPS, *G = F + SB * SB;
  auto l1 = [&](int i, int k) { return two ? L1[k * NB + i] : (i == k ? 1.0 : 0.0); };
  auto u1 = [&](int i, int k) { return two ? U1[i * NB + k] : (i == k ? 1.0 : 0.0); };
  auto l10 = [&](int i, int k) {
    return two && j1 + i < N && NB + i - k <= kl ? (double)base[(size_t)(j1 + i) + (size_t)(j0 + k) * lda] : 0.0;
  };
  auto u01 = [&](int k, int j) {
    return two && j1 + j < N && NB + j - k <= ku ? (double)base[(size_t)(j0 + k) + (size_t)(j1 + j) * lda] : 0.0;
  };
  for (int t = tid; t < NB * NB; t += 256) {
    const int j = t >> 6, i = t & 63;
    F[(size_t)j * SB + i] = L0[j * NB + i];
    F[(size_t)(NB + j) * SB + NB + i] = l1(i, j);
    F[(size_t)(NB + j) * SB + i] = 0.0;
    G[(size_t)j * SB + i] = U0[i * NB + j];
    G[(size_t)(NB + j) * SB + NB + i] = u1(i, j);
    G[(size_t)j * SB + NB + i] = 0.0;
  }
  d4v acc[2][2];
  clear(acc);  // L10 L0^-1
  product64(m0, n0, [&](int k, int i) { return l10(i, k); }, [&](int k, int n) { return L0[n * NB + k]; }, acc);
  each(m0, n0, acc, [&](int i, int n, double v) { s_t[i][n] = v; });
  __syncthreads();
  clear(acc);
  product64(m0, n0, [&](int k, int i) { return l1(i, k); }, [&](int k, int n) { return s_t[k][n]; }, acc);
  each(m0, n0, acc, [&](int i, int n, double v) { F[(size_t)n * SB + NB + i] = -v; });
  __syncthreads();
  clear(acc);  // U0^-1 U01
  product64(m0, n0, [&](int k, int i) { return U0[i * NB + k]; }, [&](int k, int n) { return u01(k, n); }, acc);
  each(m0, n0, acc, [&](int i, int n, double v) { s_t[i][n] = v; });
  __syncthreads();
  clear(acc);
  product64(m0, n0, [&](int k, int i) { return s_t[i][k]; }, [&](int k, int n) { return u1(k, n); }, acc);
  each(m0, n0, acc, [&](int i, int n, double v) { G[(size_t)(NB + n) * SB + i] = -v; });
}

// One solve step over the pair of panels at s0, by every workgroup: its 128
// values v = op w from one 128 x 128 operator (1024 threads: 128 rows x 8
// column groups), then 64 rows per workgroup of the other unknowns it couples
// to, w -= A v: the R rows below (forward) or above (UP).  Workgroup 0 writes
// v to out; w of the pair itself is only read.  All of a thread's matrix
// entries are loaded before anything waits: a step is one round of memory
// latency and two LDS reductions (64-unknown blocks with the triangle solved
// by one wave's shuffles took 13 us forward and 17 backward; this takes
// 6.1 us for 128).
template <typename T, bool UP>
__global__ __launch_bounds__(1024) void k_band_step(int N, int s0, int R, const T *__restrict__ ab,
                                                    long long off, long long lda, int band,
                                                    const double *__restrict__ ops, double *__restrict__ w,
                                                    double *__restrict__ out) {
  __shared__ double s_w[SB], s_red[16][SB], s_v[SB];
  const T *__restrict__ base = ab + off;
  const int tid = threadIdx.x, i = tid & (SB - 1), g = tid >> 7;
  const int ri = tid & 63, rg = tid >> 6;
  const double *op = ops + (size_t)(s0 / SB) * OPS + (UP ? SB * SB : 0);
  const int rr = blockIdx.x * 64 + ri, row = UP ? s0 - R + rr : s0 + SB + rr;
  double m[16], a[8];
#pragma unroll
  for (int k = 0; k < 16; k++) m[k] = op[(size_t)(16 * g + k) * SB + i];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int j = s0 + 8 * rg + k;
    a[k] = rr < R && j < N && (UP ? j - row : row - j) <= band ? (double)base[(size_t)row + (size_t)j * lda] : 0.0;
  }
  if (tid < SB) s_w[tid] = s0 + tid < N ? w[s0 + tid] : 0.0;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 16; k++) s += m[k] * s_w[16 * g + k];
  s_red[g][i] = s;
  __syncthreads();
  if (tid < SB) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) v += s_red[k][tid];
    s_v[tid] = v;
    if (blockIdx.x == 0 && s0 + tid < N) out[s0 + tid] = v;
  }
  __syncthreads();
  s = 0.0;
#pragma unroll
  for (int k = 0; k < 8; k++) s += a[k] * s_v[8 * rg + k];
  s_red[rg][ri] = s;
  __syncthreads();
  if (tid < 64 && rr < R) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 16; k++) v += s_red[k][tid];
    w[row] -= v;
  }
}

__global__ __launch_bounds__(256) void k_band_copy(int n, const double *__restrict__ a, double *__restrict__ b) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) b[i] = a[i];
}

// r = a + f b
__global__ __launch_bounds__(256) void k_band_sum(int n, const double *a, double f, const double *b, double *r) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) r[i] = a[i] + f * b[i];
}

}  // namespace

// The bandwidths of the graph.
static void band_plan(gm_ctx *c) {
  BandLU &B = c->band;
  if (B.kl >= 0) return;
  int kl = 0, ku = 0;
  for (int i = 0; i < c->N; i++)
    for (int k = c->bindx[i]; k < c->bindx[i + 1]; k++) {
      const int j = c->bindx[k];
      kl = std::max(kl, i - j);
      ku = std::max(ku, j - i);
    }
  B.kl = kl;
  B.ku = ku;
  B.ld = (long long)kl + ku + 1 + 2 * MG;
}

// The buffers that a factorisation in precision pi still needs, all of them or,
// when one does not fit, none.
static int band_buffers(gm_ctx *c, int pi) {
  BandLU &B = c->band;
  const size_t N = c->N, np = (N + NB - 1) / NB;
  struct {
    void **p;
    size_t bytes;
  } need[] = {{&B.d_ab[pi], N * B.ld * (pi ? sizeof(float) : sizeof(double))},
              {(void **)&B.d_w1, N * sizeof(double)},
              {(void **)&B.d_w2, N * sizeof(double)},
              {(void **)&B.d_ax, N * sizeof(double)},
              // (one panel beyond the last, so that an update's successor is always inside)
              {(void **)&B.d_tri, (np + 1) * TRI * sizeof(double)},
              {(void **)&B.d_ops, (np + 1) / 2 * OPS * sizeof(double)}};
  std::vector<void **> made;
  for (auto &q : need) {
    if (*q.p) continue;
    if (hipMalloc(q.p, q.bytes) == hipSuccess) {
      made.push_back(q.p);
      continue;
    }
    (void)hipGetLastError();
    *q.p = nullptr;
    for (void **m : made) {
      (void)hipFree(*m);
      *m = nullptr;
    }
    double total = 0.0;
    for (auto &r : need) total += *r.p ? 0.0 : (double)r.bytes;
    gm_set_error("banded LU needs %.1f GB (N %d, bandwidths %d / %d)", total / 1e9, c->N, B.kl, B.ku);
    return GM_ERR_ARG;
  }
  return GM_OK;
}

template <typename VT, typename T>
static int band_factor_t(gm_ctx *c, const VT *val, T *ab) {
  BandLU &B = c->band;
  const int N = c->N, kl = B.kl, ku = B.ku;
  const long long off = MG + ku, lda = B.ld - 1;
  const size_t total = (size_t)N * B.ld;
  hipStream_t s = c->stream;
  k_band_zero<T><<<4096, 256, 0, s>>>(total, ab);
  k_band_load<VT, T><<<(N + 255) / 256, 256, 0, s>>>(N, val, c->d_bindx, ab, off, lda);
  GM_HIP(hipMemsetAsync(c->d_flag + 4, 0, sizeof(int), s));
  int *d_pivflag = c->d_flag + 4;
  const int np = (N + NB - 1) / NB;
  for (int k = 0; k < np; k++) {
    const int j0 = k * NB, kb = std::min(NB, N - j0);
    const int R = std::min(kl, N - j0 - kb), C = std::min(ku, N - j0 - kb);
    const int next = std::min(NB, N - j0 - kb);
    double *tri = B.d_tri + (size_t)k * TRI;
    // a panel whose predecessor's window held its diagonal block has its triangles already
    const bool done = k > 0 && std::min(kl, N - j0) >= kb && std::min(ku, N - j0) >= kb;
    if (!done)
      gm_launch(c, GM_K_BAND_PANEL, 2.0 * kb * kb * sizeof(T), k_band_diag<T>, dim3(1), dim3(256), 0, s, j0,
                kb, (const T *)ab, off, lda, tri, d_pivflag);
    if (R <= 0 && C <= 0) continue;
    const int rt = (R + NB - 1) / NB, ct = (C + NB - 1) / NB;
    gm_launch(c, GM_K_BAND_PANEL, 2.0 * (R + C) * NB * sizeof(T), k_band_panel<T>, dim3(rt + ct), dim3(256), 0,
              s, j0, j0 + kb + R, j0 + kb + C, rt, ab, off, lda, (const double *)tri);
    if (R > 0 && C > 0)
      gm_launch(c, GM_K_BAND_UPDATE, ((double)(R + C) * NB + 2.0 * R * C) * sizeof(T), k_band_update<T>,
                dim3(rt, ct), dim3(256), 0, s, j0, j0 + kb + R, j0 + kb + C, R >= next && C >= next ? next : 0,
                ab, off, lda, tri + TRI, d_pivflag);
  }
  k_band_ops<T><<<(N + SB - 1) / SB, 256, 0, s>>>(N, (const T *)ab, off, lda, kl, ku, np,
                                                  (const double *)B.d_tri, B.d_ops);
  GM_HIP(hipGetLastError());
  int flag = 0;
  GM_HIP(hipMemcpyAsync(&flag, c->d_flag + 4, sizeof(int), hipMemcpyDeviceToHost, s));
  GM_HIP(hipStreamSynchronize(s));
  if (flag) {
    gm_set_error("zero pivot in the banded LU (no pivoting)");
    return GM_ERR_PIVOT;
  }
  return GM_OK;
}

int gm_band_factor(gm_ctx *c, const double *val, const float *val32, int prec) {
  band_plan(c);
  BandLU &B = c->band;
  const int pi = prec == GM_PREC_MIXED ? 1 : 0;
  const int rc = band_buffers(c, pi);
  if (rc) return rc;
  B.prec = pi;
  B.fresh = true;
  if (pi) {
    if (!val32) {
      gm_set_error("mixed precision needs FP32 Jacobian values");
      return GM_ERR_ARG;
    }
    return band_factor_t<float, float>(c, val32, (float *)B.d_ab[1]);
  }
  return band_factor_t<double, double>(c, val, (double *)B.d_ab[0]);
}

// out = (L U)^-1 w1, through w2; w1 is overwritten
template <typename T>
static void band_solve(gm_ctx *c, const T *ab, double *out) {
  BandLU &B = c->band;
  const int N = c->N, kl = B.kl, ku = B.ku;
  const long long off = MG + ku, lda = B.ld - 1;
  hipStream_t s = c->stream;
  const int ns = (N + SB - 1) / SB;
  for (int b = 0; b < ns; b++) {
    const int s0 = b * SB, R = std::max(0, std::min(kl, N - s0 - SB));
    const double bytes = (double)SB * R * sizeof(T) + SB * SB * 8.0 + 16.0 * (SB + R);
    gm_launch(c, GM_K_BAND_SOLVE, bytes, k_band_step<T, false>, dim3(std::max(1, (R + 63) / 64)), dim3(1024), 0,
              s, N, s0, R, ab, off, lda, kl, (const double *)B.d_ops, B.d_w1, B.d_w2);
  }
  for (int b = ns - 1; b >= 0; b--) {
    const int s0 = b * SB, R = std::min(ku, s0);
    const double bytes = (double)SB * R * sizeof(T) + SB * SB * 8.0 + 16.0 * (SB + R);
    gm_launch(c, GM_K_BAND_SOLVE, bytes, k_band_step<T, true>, dim3(std::max(1, (R + 63) / 64)), dim3(1024), 0,
              s, N, s0, R, ab, off, lda, ku, (const double *)B.d_ops, B.d_w2, out);
  }
}

// out = M^-1 in.  val: the FP64 matrix that was factored, or null.  With it the
// solve is refined once: the inverse triangles leave 1.2 to 12 times the
// residual of triangular substitution, a step of refinement the rounding of
// A x itself.  FP32 factors are not refined: their rounding outweighs the
// inverses', which are FP64.
int gm_band_apply(gm_ctx *c, const double *val, const double *in, double *out) {
  BandLU &B = c->band;
  if (B.prec < 0 || !B.d_ab[B.prec]) {
    gm_set_error("banded LU not factored");
    return GM_ERR_ARG;
  }
  hipStream_t s = c->stream;
  k_band_copy<<<1024, 256, 0, s>>>(c->N, in, B.d_w1);
  if (B.prec == 1) {
    band_solve<float>(c, (const float *)B.d_ab[1], out);
  } else {
    const double *ab = (const double *)B.d_ab[0];
    band_solve<double>(c, ab, out);
    if (val && B.fresh) {
      const int rc = gm_spmv_launch(c, val, out, B.d_ax);
      if (rc) return rc;
      k_band_sum<<<1024, 256, 0, s>>>(c->N, in, -1.0, B.d_ax, B.d_w1);
      band_solve<double>(c, ab, B.d_ax);
      k_band_sum<<<1024, 256, 0, s>>>(c->N, out, 1.0, B.d_ax, out);
    }
  }
  GM_HIP(hipGetLastError());
  return GM_OK;
}

void gm_band_free(gm_ctx *c) {
  BandLU &B = c->band;
  void *p[] = {B.d_ab[0], B.d_ab[1], B.d_w1, B.d_w2, B.d_ax, B.d_tri, B.d_ops};
  for (void *q : p)
    if (q) (void)hipFree(q);
  c->band = BandLU();
}
