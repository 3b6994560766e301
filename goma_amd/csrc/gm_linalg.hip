// Linear algebra on the MSR Jacobian: row-sum scaling, norms, SpMV,
// ILU(0) in patch order, restarted right-preconditioned GMRES.
//
// All reductions are two-stage (per-block partials, then a fixed-order sum: on
// the host, or for GMRES's projections and norms in the kernel that uses them),
// so results are bitwise reproducible run to run.
#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstring>
#include <vector>

#include "gm_launch.h"

static constexpr int RED_BLOCKS = 1024;
static constexpr int RED_THREADS = 256;

template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename T>
__device__ inline T block_sum(T v, T *sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[w] = v;
  __syncthreads();
  T s = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) s += sh[i];
  return s;  // valid on thread 0
}

// ---------------------------------------------------------------- fills
template <typename T>
__global__ void k_fill_value(T *p, long long n, T v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

int gm_zero(gm_ctx *c, double *p, long long n) {
  k_fill_value<double><<<2048, 256, 0, c->stream>>>(p, n, 0.0);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

// ---------------------------------------------------------------- row-sum scaling
// row_sum_scale_MSR (src/sl_matrix_util.c:506-600): s_i = sgn(a_ii) sum_j |a_ij|
// (sign only when |a_ii| > 1e-200); a_ij /= s_i; b_i /= s_i.  G lanes per row;
// the first G*KEEP entries of a row stay in registers between the sum and the
// scaling (one read of the matrix instead of two), longer rows re-read the
// rest.  Row sums accumulate in FP64 for either value type.
template <typename VT, int G, int KEEP>
__global__ __launch_bounds__(256) void k_row_sum_scale(int N, VT *__restrict__ a,
                                                       const int *__restrict__ bindx,
                                                       double *__restrict__ b,
                                                       double *__restrict__ scale) {
  const int gid = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (gid >= N) return;
  const int r = gid;
  const int k0 = bindx[r], k1 = bindx[r + 1];
  double s = 0.0, v[KEEP];
#pragma unroll
  for (int t = 0; t < KEEP; t++) {
    const int k = k0 + lane + G * t;
    v[t] = k < k1 ? (double)a[k] : 0.0;
    s += fabs(v[t]);
  }
  for (int k = k0 + lane + G * KEEP; k < k1; k += G) s += fabs((double)a[k]);
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  const double d = (double)a[r];
  double rs = fabs(d) + s;
  if (fabs(d) > 1.0e-200) rs = d > 0 ? rs : -rs;
#pragma unroll
  for (int t = 0; t < KEEP; t++) {
    const int k = k0 + lane + G * t;
    if (k < k1) a[k] = (VT)(v[t] / rs);
  }
  for (int k = k0 + lane + G * KEEP; k < k1; k += G) a[k] = (VT)((double)a[k] / rs);
  if (lane == 0) {
    scale[r] = rs;
    b[r] = b[r] / rs;
    a[r] = (VT)(d / rs);
  }
}

template <int G>
static void scale_g(gm_ctx *c, double *val, float *val32, double *b, double *scale) {
  const int blocks = (int)(((long long)c->N * G + 255) / 256);
  const double nnz = (double)c->nval - 1.0;
  // values read and written, the row pointers, b read and written, the scale
  const double bytes = nnz * 2.0 * (val32 ? 4.0 : 8.0) + 4.0 * (c->N + 1) + c->N * 24.0;
  constexpr int KEEP = G == 64 ? 9 : 4;  // HEX27 rows up to 576 entries, QUAD9 up to 64
  if (val32)
    gm_launch(c, GM_K_ROW_SCALE, bytes, k_row_sum_scale<float, G, KEEP>, dim3(blocks), dim3(256),
              0, c->stream, c->N, val32, c->d_bindx, b, scale);
  else
    gm_launch(c, GM_K_ROW_SCALE, bytes, k_row_sum_scale<double, G, KEEP>, dim3(blocks), dim3(256),
              0, c->stream, c->N, val, c->d_bindx, b, scale);
}

int gm_scale_launch(gm_ctx *c, double *val, float *val32, double *b, double *scale) {
  // a wave per HEX27 row (~250 entries, at most ~530), 16 lanes per QUAD9 row (~60)
  if (c->dim == 3) scale_g<64>(c, val, val32, b, scale);
  else scale_g<16>(c, val, val32, b, scale);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

// ---------------------------------------------------------------- norms
// L2_norm / Loo_norm (src/mm_sol_nonlinear.c:3177, 3320): partial sums of
// squares and partial maxima per block.
__global__ __launch_bounds__(RED_THREADS) void k_norms(const double *__restrict__ v, long long n,
                                                       double *__restrict__ part) {
  __shared__ double sh[RED_THREADS / 64];
  double s = 0.0, m = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double x = v[i];
    s += x * x;
    m = fmax(m, fabs(x));
  }
  double ss = block_sum(s, sh);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  __shared__ double shm[RED_THREADS / 64];
  if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double mm = 0.0;
    for (int i = 0; i < RED_THREADS / 64; i++) mm = fmax(mm, shm[i]);
    part[blockIdx.x] = ss;
    part[gridDim.x + blockIdx.x] = mm;
  }
}

// L2_norm_r / Loo_norm_r (src/mm_sol_nonlinear.c:3249, 3376)
__global__ __launch_bounds__(RED_THREADS) void k_corr_norms(const double *__restrict__ d,
                                                            const double *__restrict__ x,
                                                            long long n, double *__restrict__ part) {
  __shared__ double sh[RED_THREADS / 64];
  double s = 0.0, m = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double di = d[i], xi = x[i];
    s += di * di / (1 + xi * xi);
    m = fmax(m, fabs(di) / (1.0 + fabs(xi)));
  }
  double ss = block_sum(s, sh);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  __shared__ double shm[RED_THREADS / 64];
  if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double mm = 0.0;
    for (int i = 0; i < RED_THREADS / 64; i++) mm = fmax(mm, shm[i]);
    part[blockIdx.x] = ss;
    part[gridDim.x + blockIdx.x] = mm;
  }
}

static int finish_norms(gm_ctx *c, double *l2, double *loo) {
  GM_HIP(hipMemcpyAsync(c->h_red, c->d_red, 2 * RED_BLOCKS * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  GM_HIP(hipStreamSynchronize(c->stream));
  double s = 0.0, m = 0.0;
  for (int i = 0; i < RED_BLOCKS; i++) s += c->h_red[i];
  for (int i = 0; i < RED_BLOCKS; i++) m = std::max(m, c->h_red[RED_BLOCKS + i]);
  // NaN propagates through the sum; fmax drops it, so test the sum too
  *l2 = std::sqrt(s);
  *loo = std::isfinite(s) ? m : s;
  return GM_OK;
}

int gm_norms(gm_ctx *c, const double *v, long long n, double *l2, double *loo) {
  k_norms<<<RED_BLOCKS, RED_THREADS, 0, c->stream>>>(v, n, c->d_red);
  GM_HIP(hipGetLastError());
  return finish_norms(c, l2, loo);
}

int gm_corr_norms(gm_ctx *c, const double *dx, const double *x, double *l2r, double *loor) {
  k_corr_norms<<<RED_BLOCKS, RED_THREADS, 0, c->stream>>>(dx, x, c->N, c->d_red);
  GM_HIP(hipGetLastError());
  return finish_norms(c, l2r, loor);
}

// global_velocity_norm (src/mm_fill_aux.c:612-672): partial sums of x^2 over
// the velocity unknowns, the first dim of every node
__global__ __launch_bounds__(RED_THREADS) void k_velocity_sq(int num_nodes, int dim,
                                                             const int *__restrict__ fu,
                                                             const double *__restrict__ x,
                                                             double *__restrict__ part) {
  __shared__ double sh[RED_THREADS / 64];
  double s = 0.0;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < (long long)num_nodes * dim;
       t += (long long)gridDim.x * blockDim.x) {
    const int n = (int)(t / dim), a = (int)(t - (long long)n * dim);
    const double v = x[fu[n] + a];
    s += v * v;
  }
  const double ss = block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = ss;
}

int gm_velocity_norm(gm_ctx *c, const double *x, double *U) {
  k_velocity_sq<<<RED_BLOCKS, RED_THREADS, 0, c->stream>>>(c->num_nodes, c->dim, c->d_fu, x, c->d_red);
  GM_HIP(hipGetLastError());
  GM_HIP(hipMemcpyAsync(c->h_red, c->d_red, RED_BLOCKS * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  GM_HIP(hipStreamSynchronize(c->stream));
  double s = 0.0;
  for (int i = 0; i < RED_BLOCKS; i++) s += c->h_red[i];
  *U = s / ((double)c->num_nodes * c->dim);
  return GM_OK;
}

// x -= damp * dx (NLS_FULL_STEP update, src/mm_sol_nonlinear.c:2553-2557)
__global__ void k_newton_update(double *__restrict__ x, const double *__restrict__ dx, int n,
                                double damp) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    x[i] -= damp * dx[i];
}

int gm_axpy_update(gm_ctx *c, double *x, const double *dx, double damp) {
  k_newton_update<<<2048, 256, 0, c->stream>>>(x, dx, c->N, damp);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

// ---------------------------------------------------------------- MSR SpMV
// y = A x (MV_MSR, src/sl_auxutil.c:373).  G lanes per row.
template <typename VT, typename XT, typename YT, int G>
__global__ __launch_bounds__(256) void k_spmv_msr(int N, const VT *__restrict__ a,
                                                  const int *__restrict__ bindx,
                                                  const XT *__restrict__ x, YT *__restrict__ y) {
  const int r = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (r >= N) return;
  const int k0 = bindx[r], k1 = bindx[r + 1];
  // FP64 accumulation whenever the vector is FP64: an FP32 matrix times an
  // FP64 Krylov vector must not round the vector, or the Arnoldi relation
  // only holds to ~1e-7 |A||x| and GMRES stalls on ill-conditioned systems.
  using AT = typename std::conditional<sizeof(VT) == 8 || sizeof(XT) == 8, double, float>::type;
  AT s = row_dot<AT, VT, XT, G>(a, bindx, x, k0, k1, lane);
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (lane == 0) y[r] = (YT)(s + (AT)a[r] * (AT)x[r]);
}

template <typename VT, typename XT, typename YT>
static void spmv(gm_ctx *c, const VT *a, const XT *x, YT *y) {
  using AT = typename std::conditional<sizeof(VT) == 8 || sizeof(XT) == 8, double, float>::type;
  const double vec = (double)c->N * (sizeof(XT) + sizeof(YT));
  if (c->dim == 3 && c->nn_cap <= GM_NODE_CAP_MAX) {
    // HEX27: one wave per node (k_msr_nodes), values, node graph and row
    // pointers (QUAD9 rows, ~60 entries, are faster per row: 0.156 vs 0.345 ms)
    const double bytes = (double)(c->nval - 1) * sizeof(VT) +
                         4.0 * (2.0 * (c->num_nodes + 1) + c->N + c->nn_list.size()) + vec;
    size_t shm;
    const int nw = gm_msr_nodes_shape<AT>(c->nn_cap, &shm);
    gm_launch(c, GM_K_SPMV, bytes, k_msr_nodes<AT, VT, XT, YT, false>, dim3((c->num_nodes + nw - 1) / nw),
              dim3(64 * nw), shm, c->stream, c->num_nodes, c->dim, c->nv, c->nn_cap, c->d_fu, c->d_nn_ptr, c->d_nn_cols,
              c->d_bindx, a, x,
              (const XT *)nullptr, y);
    return;
  }
  // G lanes per row
  const double bytes = (double)(c->nval - 1) * (sizeof(VT) + 4) + 4.0 * (c->N + 1) + vec;
  if (c->dim == 2) {
    constexpr int G = 8;  // 2D rows hold ~50-250 entries: measured 156 vs 172 us at 256^2 (G = 16)
    const int blocks = (int)(((long long)c->N * G + 255) / 256);
    gm_launch(c, GM_K_SPMV, bytes, k_spmv_msr<VT, XT, YT, G>, dim3(blocks), dim3(256), 0, c->stream,
              c->N, a, c->d_bindx, x, y);
  } else {
    constexpr int G = 64;
    const int blocks = (int)(((long long)c->N * G + 255) / 256);
    gm_launch(c, GM_K_SPMV, bytes, k_spmv_msr<VT, XT, YT, G>, dim3(blocks), dim3(256), 0, c->stream,
              c->N, a, c->d_bindx, x, y);
  }
}

int gm_spmv_launch(gm_ctx *c, const double *val, const double *x, double *y) {
  spmv<double, double, double>(c, val, x, y);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

int gm_spmv32_launch(gm_ctx *c, const float *val, const double *x, double *y) {
  spmv<float, double, double>(c, val, x, y);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

__global__ void k_lincomb(int n, double *__restrict__ out, const double *__restrict__ a, double s,
                          const double *__restrict__ b) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    out[i] = a[i] - s * b[i];
}

__global__ void k_div_scale(int n, double *__restrict__ v, const double *__restrict__ sc) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    v[i] = v[i] / sc[i];
}

__global__ __launch_bounds__(RED_THREADS) void k_dot(int n, const double *__restrict__ a,
                                                     const double *__restrict__ b,
                                                     double *__restrict__ part) {
  __shared__ double sh[RED_THREADS / 64];
  double s = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    s += a[i] * b[i];
  double t = block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

int gm_lincomb(gm_ctx *c, double *out, const double *a, double s, const double *b) {
  k_lincomb<<<2048, 256, 0, c->stream>>>(c->N, out, a, s, b);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

// out = w0 v0 + w1 v1 + w2 v2 (null vectors and their weights skipped)
__global__ void k_lin3(int n, double *__restrict__ out, double w0, const double *__restrict__ v0,
                       double w1, const double *__restrict__ v1, double w2,
                       const double *__restrict__ v2) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double s = w0 * v0[i];
    if (v1) s += w1 * v1[i];
    if (v2) s += w2 * v2[i];
    out[i] = s;
  }
}

int gm_lin3(gm_ctx *c, double *out, double w0, const double *v0, double w1, const double *v1,
            double w2, const double *v2) {
  k_lin3<<<2048, 256, 0, c->stream>>>(c->N, out, w0, v0, w1, v1, w2, v2);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

int gm_div_scale(gm_ctx *c, double *v, const double *scale) {
  k_div_scale<<<2048, 256, 0, c->stream>>>(c->N, v, scale);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

int gm_dot(gm_ctx *c, const double *a, const double *b, double *out) {
  k_dot<<<RED_BLOCKS, RED_THREADS, 0, c->stream>>>(c->N, a, b, c->d_red);
  GM_HIP(hipGetLastError());
  GM_HIP(hipMemcpyAsync(c->h_red, c->d_red, RED_BLOCKS * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  GM_HIP(hipStreamSynchronize(c->stream));
  double s = 0.0;
  for (int i = 0; i < RED_BLOCKS; i++) s += c->h_red[i];
  *out = s;
  return GM_OK;
}

// ---------------------------------------------------------------- ILU(0)
// ILU(0) of P A P^T where P is the patch ordering.  Patches of one colour
// share no couplings, so each colour is one launch with one workgroup per
// patch.  Inside a patch the rows keep their sequential (IKJ) order of
// dependence; the host groups the patch's nodes into levels (a node depends
// on every earlier node of the patch its rows reference in L, or later node in
// U), and the workgroup walks the levels.  The arithmetic per entry is the
// sequential algorithm's; only the summation order inside a row differs.

static constexpr int ILU_MAXPATCH = 8192;  // rows of one patch held in LDS by the sweeps
static constexpr int ILU_NW = 8;           // waves per patch workgroup (sweeps)
static constexpr int ILU_D = 4;            // chunks a wave loads ahead
static constexpr int ILU_LDS = 160 * 1024; // LDS of a CU
static constexpr int ILU_FIRST = 1 << 16, ILU_LAST = 1 << 17, ILU_R8 = 1 << 18;  // chunk flags

struct IluLv {
  const int *rowptr, *col, *diag, *node_first, *node_last, *patch_row;
  const int *lv_ptr, *lv_nstart, *lv_node, *lv_rstart, *lv_row;
};

struct IluSw {
  const int *patch_row, *sp, *pre, *idx, *hptr, *halo;
  const int4 *ctl;
};

// v from the lane that the DPP control picks in the same row of 16 lanes
template <int CTRL>
__device__ inline float dpp_mov(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double dpp_mov(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// sum over 8 consecutive lanes, on all of them: quad swaps, then the half-row mirror
template <typename T>
__device__ inline T sum8(T v) {
  v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_mov<0x141>(v);  // row_half_mirror
  return v;
}

// v of lane i (the same i in every lane)
__device__ inline int lane_of(int v, int i) { return __builtin_amdgcn_readlane(v, i); }
__device__ inline float lane_of(float v, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}
__device__ inline double lane_of(double v, int i) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, i);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), i);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// The place among a node's 64 values (8 or 16 lanes a row, n unknowns) where
// its upper triangle keeps the reciprocal of diagonal k: the triangle leaves
// them free.
__host__ __device__ constexpr int ilu_recip_lane(int lsh, int n, int k) {
  return lsh == 4 ? (k << 4) + 8 + k : k < n - 1 ? ((n - 1) << 3) + k : (n - 2) << 3;
}

// x of T x = t, a node's triangle: t_i, then x_i, in all of the 1 << LSH lanes
// of row i; entry (i, k) of T in lane k of row i, unit diagonal unless UPPER.
// In the order of the sequential algorithm: x_k leaves its row through scalar
// registers, and every row takes its part of it (a finished row's is not read).
// Divisions by the reciprocal and one correction, rounded as a division; the
// reciprocals are 0 where one would leave the normal range.
template <int LSH, bool UPPER>
__device__ __forceinline__ double ilu_node_solve(double t, double T, int n) {
  const int lane = threadIdx.x & 63, i = lane >> LSH;
  double x = t;
  if (UPPER && lane_of(T, ilu_recip_lane(LSH, n, 0)) == 0.0) {
    for (int k = n - 1; k >= 0; k--) {
      const double q = __shfl(t, k << LSH) / __shfl(T, (k << LSH) + k);
      x = i == k ? q : x;
      t -= __shfl(T, (i << LSH) + k) * q;
    }
    return x;
  }
  auto step = [&](int k) {
    double q = lane_of(t, k << LSH);
    if constexpr (UPPER) {
      const double d = lane_of(T, (k << LSH) + k), r = lane_of(T, ilu_recip_lane(LSH, n, k)), q0 = q;
      q = q0 * r;
      q = fma(fma(-d, q, q0), r, q);
    }
    x = i == k ? q : x;
    double c = row_bcast(T, k);
    if constexpr (LSH == 3) c = (lane & 8) ? row_bcast(T, k + 8) : c;
    t = fma(-c, q, t);
  };
  if constexpr (UPPER) {
    if constexpr (LSH == 3) {  // five to eight unknowns
      if (n > 6) {
        if (n > 7) step(7);
        step(6);
      }
      if (n > 5) step(5);
      step(4);
      step(3);
      step(2);
      step(1);
    } else {
      if (n > 3) step(3);
      if (n > 2) step(2);
      if (n > 1) step(1);
    }
    step(0);
    return x;
  } else {
    if constexpr (LSH == 3) {
      step(0);
      step(1);
      step(2);
      step(3);
      if (n > 5) step(4);
      if (n > 6) {
        step(5);
        if (n > 7) step(6);
      }
    } else {
      if (n > 1) step(0);
      if (n > 2) step(1);
      if (n > 3) step(2);
    }
    return i == n - 1 ? t : x;
  }
}

// One triangular sweep over the patches of one colour: y = L^-1 (P b) (UPPER
// false, L unit lower) or y = U^-1 y with the unpermuted copy in out (UPPER).
// FP64 for the factors of either precision.
//
// The sweep is a chain of levels (about 65 for an 8 x 8 QUAD9 patch, 105 for
// a 4 x 4 x 4 HEX27 one) with only a few nodes each, so it is bound by the
// latency of one level, not by bandwidth.  Nothing but the solution itself
// may therefore sit on that chain: the entries come from streams laid out in
// the order they are used, one per wave, and are loaded ILU_D chunks ahead
// into registers; the patch's rows and the rows of other patches it reads (its
// halo) are in LDS; and a node's small triangle is solved in registers
// (ilu_node_solve).  A level is then LDS reads of y, a few FMAs, one row
// reduction, two to four dependent steps of the triangle, an LDS write and a
// barrier.
// A chunk is CE entries per lane of one node: four rows of 16 lanes, or eight
// rows of 8 lanes (nodes of more than four unknowns).  LDSH: every patch's
// halo is in LDS; otherwise a load of y may stand in the chain, and the wait
// for it takes the loads in flight along.  A wave without a node in a level
// only takes its barrier (ctl.z).
// Measured on the 32 x 32 QUAD9 cavity (four patches a colour, 62 levels): 35
// us a launch forward (0.57 us a level) and 43 backward (0.70); with the entries
// read through the CSR factors level by level, two barriers a level and the
// triangle solved row after row through LDS it took 190 and 226.  With the
// node's inverse triangle multiplied into its entries, 29 us; but on saddle
// points its residual was up to 100,000 times the substitution's.
template <typename BT, typename OT, int CE, bool UPPER, bool LDSH>
__global__ __launch_bounds__(ILU_NW * 64) void k_ilu_sweep(IluSw S, const double *__restrict__ val,
                                                           const double *__restrict__ tri, int patch0,
                                                           const int *__restrict__ perm,
                                                           const BT *__restrict__ b, double *y,
                                                           OT *__restrict__ out) {
  extern __shared__ double s_y[];
  const int P = patch0 + blockIdx.x;
  const int r0 = S.patch_row[P], nr = S.patch_row[P + 1] - r0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = S.sp[P * ILU_NW + w], c1 = S.sp[P * ILU_NW + w + 1];
  const int npre = S.pre[P * ILU_NW + w];

  double rv[ILU_D][CE], rt[ILU_D];
  int rx[ILU_D][CE];
  int4 rc[ILU_D];
  // The control words go through vector registers (vz is 0, but not known to
  // be): a scalar load in flight would have to be waited for at every LDS wait.
  const int vz = (tid >> 6) - w;
  auto fetch = [&](int d, int c) {
    rc[d] = S.ctl[c + vz];
    const size_t at = (size_t)c * (64 * CE) + lane;
#pragma unroll
    for (int e = 0; e < CE; e++) {
      rv[d][e] = val[at + 64 * e];
      rx[d][e] = S.idx[at + 64 * e];
    }
    rt[d] = tri[(size_t)c * 64 + lane];
  };
#pragma unroll
  for (int d = 0; d < ILU_D; d++) fetch(d, c0 + d);  // the streams end in ILU_D spare chunks

  for (int i = tid; i < nr; i += ILU_NW * 64) s_y[i] = UPPER ? y[r0 + i] : (double)b[perm[r0 + i]];
  const int h0 = S.hptr[P], nh = S.hptr[P + 1] - h0;
  for (int i = tid; i < nh; i += ILU_NW * 64) s_y[nr + i] = y[S.halo[h0 + i]];
  auto level_end = [&]() {  // the solution in LDS, nothing of the loads in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  level_end();
  for (int k = 0; k < npre; k++) level_end();

  double acc = 0;
  for (int c = c0; c < c1; c += ILU_D) {
#pragma unroll
    for (int d = 0; d < ILU_D; d++) {
      const int flags = __builtin_amdgcn_readfirstlane(rc[d].x), n = __builtin_amdgcn_readfirstlane(rc[d].y);
      const int bars = __builtin_amdgcn_readfirstlane(rc[d].z);
      const int lsh = (flags & ILU_R8) ? 3 : 4;  // log2 of the lanes of a row
      const int row = flags & (ILU_FIRST - 1), k = lane & ((1 << lsh) - 1);
      const int i = lane >> lsh;
      const double T = rt[d];
      double s = acc;
      if (flags & ILU_FIRST) s = k == 0 && i < n ? s_y[row + i] : 0.0;
#pragma unroll
      for (int e = 0; e < CE; e++) {
        const int j = rx[d][e];
        s -= rv[d][e] * (LDSH || j >= 0 ? s_y[j] : y[~j]);
      }
      acc = s;
      fetch(d, c + d + ILU_D);
      if (flags & ILU_LAST) {
        s = sum8(s);
        if (lsh == 4) {
          s += dpp_mov<0x140>(s);  // row_mirror: the other half of the 16 lanes
          s = ilu_node_solve<4, UPPER>(s, T, n);
        } else {
          s = ilu_node_solve<3, UPPER>(s, T, n);
        }
        if (k == 0 && i < n) s_y[row + i] = s;
      }
      for (int q = 0; q < bars; q++) level_end();
    }
  }
  level_end();
  for (int i = tid; i < nr; i += ILU_NW * 64) {
    const double v = s_y[i];
    y[r0 + i] = v;
    if (UPPER) out[perm[r0 + i]] = (OT)v;
  }
}

// Each node's triangle of the factors (at most 8 x 8) as ilu_node_solve takes
// it, at the place of the node's last chunk; a wave per node.
template <typename VT, bool UPPER>
__global__ __launch_bounds__(256) void k_ilu_node_tri(int nodes, const int2 *__restrict__ node,
                                                      const int *__restrict__ node_last,
                                                      const int *__restrict__ rowptr,
                                                      const int *__restrict__ col,
                                                      const int *__restrict__ diag,
                                                      const VT *__restrict__ lu, double *__restrict__ tri) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= nodes) return;
  const int nf = node[t].x, n = node_last[nf] - nf + 1, lsh = n > 4 ? 3 : 4;
  const int i = lane >> lsh, k = lane & ((1 << lsh) - 1);
  double v = 0.0;
  if (i < n && k < n) {
    const int r = nf + i, cc = nf + k, d = diag[r];
    if (!UPPER) {
      for (int p = d - 1; p >= rowptr[r] && col[p] >= cc; p--)
        if (col[p] == cc) v = (double)lu[p];
    } else {
      for (int p = d; p < rowptr[r + 1] && col[p] <= cc; p++)
        if (col[p] == cc) v = (double)lu[p];
    }
  }
  if (UPPER) {
    bool normal = true;
    for (int q = 0; q < n; q++) {
      const double r = 1.0 / (double)lu[diag[nf + q]];
      normal = normal && fabs(r) >= 0x1p-1021 && fabs(r) <= 0x1p1021;
      if (lane == ilu_recip_lane(lsh, n, q)) v = r;
    }
    if (!normal)
      for (int q = 0; q < n; q++)
        if (lane == ilu_recip_lane(lsh, n, q)) v = 0.0;
  }
  tri[(size_t)node[t].y * 64 + lane] = v;
}

// The factors' off-node entries in stream order, zero where a chunk is padded.
template <typename VT>
__global__ __launch_bounds__(256) void k_ilu_pack(long long n, const int *__restrict__ src,
                                                  const VT *__restrict__ lu, double *__restrict__ val) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL)
    val[i] = src[i] >= 0 ? (double)lu[src[i]] : 0.0;
}

static IluLv lv_args(const IluPlan &P) {
  IluLv S;
  S.rowptr = P.d_rowptr;
  S.col = P.d_col;
  S.diag = P.d_diag;
  S.node_first = P.d_node_first;
  S.node_last = P.d_node_last;
  S.patch_row = P.d_patch_row;
  S.lv_ptr = P.d_lv_ptr;
  S.lv_nstart = P.d_lv_nstart;
  S.lv_node = P.d_lv_node;
  S.lv_rstart = P.d_lv_rstart;
  S.lv_row = P.d_lv_row;
  return S;
}

// IKJ elimination of row r by the pivot rows whose column lies in [kb, ke),
// one wavefront per row, the row staged in LDS.  The pivot rows follow one
// another through the row, so what a step waits for is what counts: up to 64
// pivot rows' places and diagonals are fetched together, a lane each, and a
// pivot row's entries a step ahead; a step is then the search of its columns
// and the update, both in LDS (a patch colour of the 32 x 32 cavity, 11,500
// unknowns: 1.8 ms against 3.5 with four dependent loads from memory in
// every step and half the waves).
template <typename VT>
__device__ inline void ilu_row_eliminate(const IluLv &S, VT *lu, int r, int kb, int ke, int *s_col,
                                         VT *s_val, int *flag) {
  const int lane = threadIdx.x & 63;
  const int b = S.rowptr[r], len = S.rowptr[r + 1] - b, dpos = S.diag[r] - b;
  for (int t = lane; t < len; t += 64) {
    s_col[t] = S.col[b + t];
    s_val[t] = lu[b + t];
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  for (int q0 = 0; q0 < dpos; q0 += 64) {
    const int t = q0 + lane, k = t < dpos ? s_col[t] : -1;
    const bool in = k >= kb && k < ke;  // (a run of the ascending columns)
    const unsigned long long mask = __ballot(in);
    if (!mask) continue;
    int dk = 0, kend = 0;
    VT piv = (VT)1;
    if (in) {
      dk = S.diag[k];
      kend = S.rowptr[k + 1];
      piv = lu[dk];
    }
    const int first = __ffsll(mask) - 1, last = 63 - __clzll((long long)mask);
    auto fetch = [&](int i, int *j, VT *u) {
      const int jj = lane_of(dk, i) + 1 + lane;
      *j = -1;
      *u = (VT)0;
      if (jj < lane_of(kend, i)) {
        *j = S.col[jj];
        *u = lu[jj];
      }
    };
    int jn;
    VT un;
    fetch(first, &jn, &un);
    for (int i = first; i <= last; i++) {
      const int j0 = jn, kk = q0 + i;
      const VT u0 = un;
      if (i < last) fetch(i + 1, &jn, &un);
      const VT l = s_val[kk] / lane_of(piv, i);
      __builtin_amdgcn_wave_barrier();
      if (lane == 0) s_val[kk] = l;
      const int n = len - kk - 1;
      auto apply = [&](int j, VT u) {  // the entry of column j, if the row has one
        int at = kk + 1;
        for (int step = n ? 1 << (31 - __clz(n)) : 0; step; step >>= 1)
          if (at + step <= len && s_col[at + step - 1] < j) at += step;
        if (j >= 0 && at < len && s_col[at] == j) s_val[at] -= l * u;
      };
      apply(j0, u0);
      const int e = lane_of(kend, i);
      for (int jj = lane_of(dk, i) + 65 + lane; jj < e; jj += 64) apply(S.col[jj], lu[jj]);
      __builtin_amdgcn_wave_barrier();
      __threadfence_block();
    }
  }
  for (int t = lane; t < len; t += 64) lu[b + t] = s_val[t];
  if (lane == 0 && ke > r && s_val[dpos] == (VT)0) atomicOr(flag + 2, 1);
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
}

// LDS: cap (the longest row) values and columns per wave
template <typename VT>
__global__ __launch_bounds__(1024) void k_ilu_factor(IluLv S, VT *lu, int patch0, int cap, int *flag) {
  extern __shared__ double s_rows[];
  const int P = patch0 + blockIdx.x;
  const int w = threadIdx.x >> 6, NW = blockDim.x >> 6;
  VT *s_val = (VT *)s_rows + (size_t)w * cap;
  int *s_col = (int *)((VT *)s_rows + (size_t)NW * cap) + (size_t)w * cap;
  for (int l = S.lv_ptr[P]; l < S.lv_ptr[P + 1]; l++) {
    // rows of the level against pivot rows outside their own node
    for (int k = S.lv_rstart[l] + w; k < S.lv_rstart[l + 1]; k += NW) {
      const int r = S.lv_row[k];
      ilu_row_eliminate<VT>(S, lu, r, 0, S.node_first[r], s_col, s_val, flag);
    }
    __syncthreads();
    // each node's rows against the node's earlier rows, in order
    for (int k = S.lv_nstart[l] + w; k < S.lv_nstart[l + 1]; k += NW) {
      const int nf = S.lv_node[k];
      const int nl = S.node_last[nf];
      for (int r = nf; r <= nl; r++) ilu_row_eliminate<VT>(S, lu, r, nf, r + 1, s_col, s_val, flag);
    }
    __syncthreads();
  }
}

template <typename VT>
static int ilu_factor_colour(gm_ctx *c, VT *lu, int p0, int cnt) {
  IluPlan &P = c->ilu;
  const size_t wave = (size_t)P.maxrow * (sizeof(VT) + sizeof(int));
  // 16 waves where their rows fit (2D, HEX27), 8 beyond
  const int nw = 16 * wave <= (size_t)ILU_LDS ? 16 : 8;
  if (nw * wave > 64 * 1024)
    GM_HIP(hipFuncSetAttribute((const void *)k_ilu_factor<VT>, hipFuncAttributeMaxDynamicSharedMemorySize, ILU_LDS));
  gm_launch(c, GM_K_ILU_FACT, 0.0, k_ilu_factor<VT>, dim3(cnt), dim3(64 * nw), nw * wave, c->stream, lv_args(P), lu, p0,
            P.maxrow, c->d_flag);
  return GM_OK;
}

// gather MSR values into the permuted CSR
template <typename VT, typename DT>
__global__ void k_ilu_gather(long long n, const int *__restrict__ src, const VT *__restrict__ a,
                         DT *__restrict__ lu) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    lu[i] = (DT)a[src[i]];
}

static void free_plan(IluPlan &P) {
  void *ptrs[] = {P.d_perm, P.d_rowptr, P.d_col, P.d_diag, P.d_src, P.d_patch_row, P.d_lu,
                  P.d_lu32, P.d_y, P.d_node_first, P.d_node_last,
                  P.d_lv_ptr, P.d_lv_nstart, P.d_lv_node, P.d_lv_rstart, P.d_lv_row};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  for (const IluStream &T : P.sweep) {
    void *q[] = {T.d_sp, T.d_pre, T.d_ctl, T.d_idx, T.d_src, T.d_node, T.d_hptr, T.d_halo,
                 T.d_val, T.d_tri};
    for (void *p : q)
      if (p) (void)hipFree(p);
  }
  P = IluPlan();
}

template <typename T>
static int up(T **d, const std::vector<T> &h) {
  GM_HIP(hipMalloc(d, std::max<size_t>(h.size(), 1) * sizeof(T)));
  if (!h.empty()) GM_HIP(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  return GM_OK;
}

struct IluHost {
  const std::vector<int> &rowptr, &col, &diag, &node_first, &node_last;
};

// The per-wave chunk streams of one sweep (k_ilu_sweep): each level's nodes
// dealt to the waves in turn, a node's couplings to the patch's other nodes
// (or to rows outside the patch) cut into chunks of CE entries per lane.
static int build_stream(IluPlan &P, const IluHost &H, bool upper, int CE,
                        const std::vector<int> &lv_ptr, const std::vector<int> &lv_nstart,
                        const std::vector<int> &lv_node) {
  IluStream &T = P.sweep[upper ? 1 : 0];
  const int np = P.npatch;
  // off-node entries of row r: [first, last) of its CSR range
  auto range = [&](int r, int *a, int *e) {
    const int nf = H.node_first[r], nl = H.node_last[nf];
    if (!upper) {
      *a = H.rowptr[r];
      *e = H.diag[r];
      while (*e > *a && H.col[*e - 1] >= nf) (*e)--;
    } else {
      *a = H.diag[r] + 1;
      *e = H.rowptr[r + 1];
      while (*a < *e && H.col[*a] <= nl) (*a)++;
    }
  };
  // the off-node columns of a node's rows, ascending
  auto columns = [&](int nf, std::vector<int> &u) {
    u.clear();
    for (int r = nf; r <= H.node_last[nf]; r++) {
      int a, e;
      range(r, &a, &e);
      u.insert(u.end(), H.col.begin() + a, H.col.begin() + e);
    }
    std::sort(u.begin(), u.end());
    u.erase(std::unique(u.begin(), u.end()), u.end());
  };
  // chunks of each node, in level order
  std::vector<int> nchunk(lv_node.size());
#pragma omp parallel
  {
    std::vector<int> u;
#pragma omp for schedule(static)
    for (size_t k = 0; k < lv_node.size(); k++) {
      const int nf = lv_node[k], per = (H.node_last[nf] - nf + 1 > 4 ? 8 : 16) * CE;
      columns(nf, u);
      nchunk[k] = std::max(1, ((int)u.size() + per - 1) / per);
    }
  }
  // stream lengths, rounded up to whole groups of ILU_D chunks
  std::vector<int> sp((size_t)np * ILU_NW + 1, 0), pre((size_t)np * ILU_NW, 0);
  for (int p = 0; p < np; p++)
    for (int l = lv_ptr[p]; l < lv_ptr[p + 1]; l++)
      for (int k = lv_nstart[l]; k < lv_nstart[l + 1]; k++)
        sp[(size_t)p * ILU_NW + (k - lv_nstart[l]) % ILU_NW + 1] += nchunk[k];
  for (size_t i = 1; i < sp.size(); i++) {
    const long long len = (sp[i] + ILU_D - 1) / ILU_D * ILU_D + (long long)sp[i - 1];
    if (len + ILU_D >= (1LL << 31)) {
      gm_set_error("ILU sweep streams too long");
      return GM_ERR_ARG;
    }
    sp[i] = (int)len;
  }
  T.chunks = (long long)sp.back() + ILU_D;
  T.entries = T.chunks * 64 * CE;
  T.nodes = (int)lv_node.size();
  std::vector<int4> ctl(T.chunks, make_int4(0, 0, 0, 0));
  std::vector<int> idx(T.entries, 0), src(T.entries, -1);
  std::vector<int2> node(lv_node.size());
  std::vector<std::vector<int>> halo(np);
  T.lds_rows = 1;
#pragma omp parallel for schedule(dynamic, 1)
  for (int p = 0; p < np; p++) {
    const int r0 = P.patch_row[p], r1 = P.patch_row[p + 1];
    // rows outside the patch that it reads: in LDS behind its own when they fit
    std::vector<int> &h = halo[p], u;
    for (int k = lv_nstart[lv_ptr[p]]; k < lv_nstart[lv_ptr[p + 1]]; k++)
      for (int r = lv_node[k]; r <= H.node_last[lv_node[k]]; r++) {
        int a, e;
        range(r, &a, &e);
        for (int t = a; t < e; t++)
          if (H.col[t] < r0 || H.col[t] >= r1) h.push_back(H.col[t]);
      }
    std::sort(h.begin(), h.end());
    h.erase(std::unique(h.begin(), h.end()), h.end());
    const bool fits = (size_t)(r1 - r0 + h.size()) * sizeof(double) <= (size_t)ILU_LDS;
    if (!fits) h.clear();
    int at[ILU_NW];
    int last[ILU_NW];
    for (int w = 0; w < ILU_NW; w++) {
      at[w] = sp[(size_t)p * ILU_NW + w];
      last[w] = -1;
    }
    for (int l = lv_ptr[p]; l < lv_ptr[p + 1]; l++) {
      for (int k = lv_nstart[l]; k < lv_nstart[l + 1]; k++) {
        const int w = (k - lv_nstart[l]) % ILU_NW;
        const int nf = lv_node[k], n = H.node_last[nf] - nf + 1, lanes = n > 4 ? 8 : 16;
        columns(nf, u);
        for (int i = 0; i < n; i++) {
          int t, e;
          range(nf + i, &t, &e);
          for (int q = 0; q < (int)u.size(); q++) {
            const int ch = at[w] + q / (lanes * CE), rem = q % (lanes * CE), cc = u[q];
            const size_t pos = (size_t)ch * 64 * CE + (size_t)(rem / lanes) * 64 + i * lanes + rem % lanes;
            if (t < e && H.col[t] == cc) src[pos] = t++;
            if (cc >= r0 && cc < r1) idx[pos] = cc - r0;
            else if (fits)
              idx[pos] = r1 - r0 + (int)(std::lower_bound(h.begin(), h.end(), cc) - h.begin());
            else idx[pos] = ~cc;
          }
        }
        for (int ch = 0; ch < nchunk[k]; ch++) {
          int4 &ct = ctl[at[w] + ch];
          ct.x = (nf - r0) | (ch == 0 ? ILU_FIRST : 0) | (ch == nchunk[k] - 1 ? ILU_LAST : 0) |
                 (n > 4 ? ILU_R8 : 0);
          ct.y = n;
        }
        at[w] += nchunk[k];
        last[w] = at[w] - 1;
        node[k] = make_int2(nf, last[w]);
      }
      for (int w = 0; w < ILU_NW; w++) {
        if (last[w] < 0) pre[(size_t)p * ILU_NW + w]++;
        else ctl[last[w]].z++;
      }
    }
#pragma omp critical
    {
      T.lds_rows = std::max(T.lds_rows, r1 - r0 + (int)h.size());
      T.halo_lds = T.halo_lds && fits;
    }
  }
  std::vector<int> hptr(np + 1, 0), hall;
  for (int p = 0; p < np; p++) {
    hall.insert(hall.end(), halo[p].begin(), halo[p].end());
    hptr[p + 1] = (int)hall.size();
  }
  int rc;
  if ((rc = up(&T.d_sp, sp)) || (rc = up(&T.d_pre, pre)) || (rc = up(&T.d_ctl, ctl)) ||
      (rc = up(&T.d_idx, idx)) || (rc = up(&T.d_src, src)) || (rc = up(&T.d_node, node)) ||
      (rc = up(&T.d_hptr, hptr)) || (rc = up(&T.d_halo, hall)))
    return rc;
  return GM_OK;
}

int gm_ilu_plan(gm_ctx *c, int bins) {
  IluPlan &P = c->ilu;
  if (P.bins == bins) return GM_OK;
  if (P.d_perm) free_plan(P);
  std::vector<int> cptr;
  int ncol = gm_patch_order(c, bins, P.perm, cptr, P.patch_row);
  if (ncol < 0) return ncol;
  P.ncol = ncol;
  P.colour_ptr = cptr;
  P.npatch = (int)P.patch_row.size() - 1;
  for (int p = 0; p < P.npatch; p++)
    if (P.patch_row[p + 1] - P.patch_row[p] > ILU_MAXPATCH) {
      gm_set_error("ILU patch with %d rows exceeds %d; use more patch bins",
                   P.patch_row[p + 1] - P.patch_row[p], ILU_MAXPATCH);
      return GM_ERR_ARG;
    }
  const int N = c->N;
  std::vector<int> iperm(N);
  for (int i = 0; i < N; i++) iperm[P.perm[i]] = i;
  std::vector<int> rowptr(N + 1, 0);
  for (int r = 0; r < N; r++) {
    const int i = P.perm[r];
    rowptr[r + 1] = 1 + c->bindx[i + 1] - c->bindx[i];
  }
  for (int r = 0; r < N; r++) rowptr[r + 1] += rowptr[r];
  const long long nnz = rowptr[N];
  P.nnz = nnz;
  std::vector<int> col(nnz), src(nnz), diag(N);
#pragma omp parallel
  {
    std::vector<std::pair<int, int>> tmp;
#pragma omp for schedule(dynamic, 4096)
    for (int r = 0; r < N; r++) {
      const int i = P.perm[r];
      tmp.clear();
      tmp.emplace_back(r, i);
      for (int k = c->bindx[i]; k < c->bindx[i + 1]; k++) tmp.emplace_back(iperm[c->bindx[k]], k);
      std::sort(tmp.begin(), tmp.end());
      const int b = rowptr[r];
      for (size_t t = 0; t < tmp.size(); t++) {
        col[b + t] = tmp[t].first;
        src[b + t] = tmp[t].second;
        if (tmp[t].first == r) diag[r] = b + (int)t;
      }
    }
  }
  P.maxrow = 1;
  for (int r = 0; r < N; r++) P.maxrow = std::max(P.maxrow, rowptr[r + 1] - rowptr[r]);
  if (P.maxrow > GM_MAXROW) {
    gm_set_error("Jacobian row longer than %d", GM_MAXROW);
    return GM_ERR_ARG;
  }
  // nodes in permuted numbering: the unknowns of a mesh node stay contiguous
  std::vector<int> node_first(N), node_last(N);
  {
    std::vector<int> node_of(N);
    for (int n = 0; n < c->num_nodes; n++)
      for (int u = c->first_unknown[n]; u < c->first_unknown[n + 1]; u++) node_of[u] = n;
    int r = 0;
    while (r < N) {
      const int n = node_of[P.perm[r]];
      const int cnt = c->first_unknown[n + 1] - c->first_unknown[n];
      for (int k = 0; k < cnt; k++) {
        node_first[r + k] = r;
        node_last[r + k] = r + cnt - 1;
      }
      r += cnt;
    }
  }
  // level schedules per patch (0: forward / factorisation, 1: backward)
  std::vector<int> lv_ptr[2], lv_nstart[2], lv_node[2], lv_rstart[2], lv_row[2];
  {
    std::vector<int> level(N, 0);
    for (int u = 0; u < 2; u++) {
      lv_ptr[u].assign(1, 0);
      lv_nstart[u].assign(1, 0);
      lv_rstart[u].assign(1, 0);
      for (int p = 0; p < P.npatch; p++) {
        const int r0 = P.patch_row[p], r1 = P.patch_row[p + 1];
        std::vector<int> nodes;
        for (int r = r0; r < r1; r = node_last[r] + 1) nodes.push_back(r);
        int maxlev = -1;
        if (u == 0) {
          for (int nf : nodes) {
            int lv = 0;
            for (int r = nf; r <= node_last[nf]; r++)
              for (int t = rowptr[r]; t < diag[r]; t++) {
                const int cc = col[t];
                if (cc >= r0 && cc < nf) lv = std::max(lv, level[node_first[cc]] + 1);
              }
            level[nf] = lv;
            maxlev = std::max(maxlev, lv);
          }
        } else {
          for (auto it = nodes.rbegin(); it != nodes.rend(); ++it) {
            const int nf = *it, nl = node_last[nf];
            int lv = 0;
            for (int r = nf; r <= nl; r++)
              for (int t = diag[r] + 1; t < rowptr[r + 1]; t++) {
                const int cc = col[t];
                if (cc > nl && cc < r1) lv = std::max(lv, level[node_first[cc]] + 1);
              }
            level[nf] = lv;
            maxlev = std::max(maxlev, lv);
          }
        }
        std::vector<std::vector<int>> byl(maxlev + 1);
        for (int nf : nodes) byl[level[nf]].push_back(nf);
        for (int lv = 0; lv <= maxlev; lv++) {
          for (int nf : byl[lv]) {
            lv_node[u].push_back(nf);
            for (int r = nf; r <= node_last[nf]; r++) lv_row[u].push_back(r);
          }
          lv_nstart[u].push_back((int)lv_node[u].size());
          lv_rstart[u].push_back((int)lv_row[u].size());
        }
        lv_ptr[u].push_back((int)lv_nstart[u].size() - 1);
      }
    }
  }
  P.levels = (int)lv_ptr[0].back();
  // per colour: rows and strictly-lower / upper (incl. diagonal) entries, for
  // the algorithmic-byte counts of the sweeps
  P.col_rows.assign(ncol, 0);
  P.col_nnzL.assign(ncol, 0);
  P.col_nnzU.assign(ncol, 0);
  for (int col = 0; col < ncol; col++) {
    const int ra = P.patch_row[P.colour_ptr[col]], rb = P.patch_row[P.colour_ptr[col + 1]];
    P.col_rows[col] = rb - ra;
    for (int r = ra; r < rb; r++) {
      P.col_nnzL[col] += diag[r] - rowptr[r];
      P.col_nnzU[col] += rowptr[r + 1] - diag[r];
    }
  }
  int rc;
  if ((rc = up(&P.d_perm, P.perm)) || (rc = up(&P.d_rowptr, rowptr)) || (rc = up(&P.d_col, col)) ||
      (rc = up(&P.d_diag, diag)) || (rc = up(&P.d_src, src)) || (rc = up(&P.d_patch_row, P.patch_row)) ||
      (rc = up(&P.d_node_first, node_first)) || (rc = up(&P.d_node_last, node_last)))
    return rc;
  if ((rc = up(&P.d_lv_ptr, lv_ptr[0])) || (rc = up(&P.d_lv_nstart, lv_nstart[0])) ||
      (rc = up(&P.d_lv_node, lv_node[0])) || (rc = up(&P.d_lv_rstart, lv_rstart[0])) ||
      (rc = up(&P.d_lv_row, lv_row[0])))
    return rc;
  const IluHost H{rowptr, col, diag, node_first, node_last};
  for (int u = 0; u < 2; u++)
    if ((rc = build_stream(P, H, u == 1, c->dim == 2 ? 3 : 4, lv_ptr[u], lv_nstart[u], lv_node[u])))
      return rc;
  GM_HIP(hipMalloc(&P.d_lu, nnz * sizeof(double)));
  GM_HIP(hipMalloc(&P.d_y, N * sizeof(double)));
  P.bins = bins;
  return GM_OK;
}

// the sweeps' streams from the factors: entries and triangles
template <typename VT>
static void ilu_streams(gm_ctx *c, const VT *lu) {
  IluPlan &P = c->ilu;
  for (int u = 0; u < 2; u++) {
    IluStream &T = P.sweep[u];
    auto kern = u ? k_ilu_node_tri<VT, true> : k_ilu_node_tri<VT, false>;
    kern<<<(T.nodes + 3) / 4, 256, 0, c->stream>>>(T.nodes, T.d_node, P.d_node_last, P.d_rowptr,
                                                   P.d_col, P.d_diag, lu, T.d_tri);
    k_ilu_pack<VT><<<(int)std::min<long long>((T.entries + 255) / 256, 16384), 256, 0, c->stream>>>(
        T.entries, T.d_src, lu, T.d_val);
  }
}

// the kernel of sweep u
template <typename RT, typename ZT, int CE>
static auto ilu_kernel(const IluStream &T, int u) {
  return T.halo_lds ? (u ? k_ilu_sweep<RT, ZT, CE, true, true> : k_ilu_sweep<RT, ZT, CE, false, true>)
                    : (u ? k_ilu_sweep<RT, ZT, CE, true, false> : k_ilu_sweep<RT, ZT, CE, false, false>);
}

// Allows the sweeps the LDS they take, before the factorisation that they apply:
// the application itself has no call that fails.  (A kernel's limit is the
// process's: every context sets the same.)
static int ilu_sweep_lds(gm_ctx *c) {
  for (int u = 0; u < 2; u++) {
    const IluStream &T = c->ilu.sweep[u];
    if ((size_t)T.lds_rows * sizeof(double) <= 64 * 1024) continue;
    auto kern = c->dim == 2 ? ilu_kernel<double, double, 3>(T, u) : ilu_kernel<double, double, 4>(T, u);
    GM_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, ILU_LDS));
  }
  return GM_OK;
}

// factorise the (scaled) Jacobian; prec 0: FP64 values, 1: FP32 values
int gm_ilu_factor(gm_ctx *c, const double *val, const float *val32, int prec) {
  IluPlan &P = c->ilu;
  if (prec == GM_PREC_MIXED && !P.d_lu32) GM_HIP(hipMalloc(&P.d_lu32, P.nnz * sizeof(float)));
  const int pi = prec == GM_PREC_MIXED ? 1 : 0;
  for (IluStream &T : P.sweep) {
    if (!T.d_tri) GM_HIP(hipMalloc(&T.d_tri, (size_t)T.chunks * 64 * sizeof(double)));
    if (!T.d_val) GM_HIP(hipMalloc(&T.d_val, (size_t)T.entries * sizeof(double)));
  }
  int rc = ilu_sweep_lds(c);
  if (rc) return rc;
  GM_HIP(hipMemsetAsync(c->d_flag + 2, 0, sizeof(int), c->stream));
  if (prec == GM_PREC_MIXED) {
    if (val32) k_ilu_gather<float, float><<<4096, 256, 0, c->stream>>>(P.nnz, P.d_src, val32, P.d_lu32);
    else k_ilu_gather<double, float><<<4096, 256, 0, c->stream>>>(P.nnz, P.d_src, val, P.d_lu32);
  } else {
    k_ilu_gather<double, double><<<4096, 256, 0, c->stream>>>(P.nnz, P.d_src, val, P.d_lu);
  }
  for (int col = 0; col < P.ncol; col++) {
    const int p0 = P.colour_ptr[col], cnt = P.colour_ptr[col + 1] - p0;
    if (!cnt) continue;
    rc = pi ? ilu_factor_colour(c, P.d_lu32, p0, cnt) : ilu_factor_colour(c, P.d_lu, p0, cnt);
    if (rc) return rc;
  }
  if (prec == GM_PREC_MIXED) ilu_streams<float>(c, P.d_lu32);
  else ilu_streams<double>(c, P.d_lu);
  GM_HIP(hipGetLastError());
  int flag = 0;
  GM_HIP(hipMemcpyAsync(&flag, c->d_flag + 2, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  GM_HIP(hipStreamSynchronize(c->stream));
  if (flag) {
    gm_set_error("zero pivot in ILU(0)");
    return GM_ERR_PIVOT;
  }
  return GM_OK;
}

// z = M^-1 r  (r, z unpermuted)
template <typename RT, typename ZT, int CE>
static void ilu_apply_ce(gm_ctx *c, const RT *r, ZT *z) {
  IluPlan &P = c->ilu;
  for (int u = 0; u < 2; u++) {
    const IluStream &T = P.sweep[u];
    auto kern = ilu_kernel<RT, ZT, CE>(T, u);
    const size_t lds = (size_t)T.lds_rows * sizeof(double);
    const IluSw S{P.d_patch_row, T.d_sp, T.d_pre, T.d_idx, T.d_hptr, T.d_halo, T.d_ctl};
    for (int k = 0; k < P.ncol; k++) {
      const int col = u ? P.ncol - 1 - k : k;
      const int p0 = P.colour_ptr[col], cnt = P.colour_ptr[col + 1] - p0;
      if (!cnt) continue;
      // values + columns of the triangle, the permutation, the input (gathered)
      // and output vectors
      const double bytes = (double)(u ? P.col_nnzU[col] : P.col_nnzL[col]) * 12.0 +
                           (double)P.col_rows[col] * (4 + (u ? 16 + sizeof(ZT) : 8 + sizeof(RT)));
      gm_launch(c, u ? GM_K_ILU_UPPER : GM_K_ILU_LOWER, bytes, kern, dim3(cnt), dim3(ILU_NW * 64), lds,
                c->stream, S, (const double *)T.d_val, (const double *)T.d_tri, p0, (const int *)P.d_perm, r, P.d_y, z);
    }
  }
}

template <typename RT, typename ZT>
static void ilu_apply(gm_ctx *c, const RT *r, ZT *z) {
  if (c->dim == 2) ilu_apply_ce<RT, ZT, 3>(c, r, z);
  else ilu_apply_ce<RT, ZT, 4>(c, r, z);
}

// The orthogonalisation of w against V[0 .. nk): three launches without the
// host in between, each of the last two finishing the sums that the one before
// left per block, so that nothing is copied and the host waits once an
// iteration.  With four copies, two waits and sums over the blocks on the host
// an iteration of 11,500 unknowns cost 85 us more; k_mdot took 20 us there with
// one vector after the other, 5.4 with eight at a time.

constexpr int DOT_T = 8;  // vectors per block of k_mdot

constexpr int DOT_PARTS = 4096;  // most partial sums, tiles DOT_T chunks
static_assert(GM_KSPACE_MAX + 1 <= DOT_PARTS, "a partial sum for every vector and for w.w");

// most blocks of k_orth_update and k_normalise, which each add up the sums
// before them: four per CU keep enough loads in flight (4.1 million unknowns:
// 50 and 12.8 us a call, 5.3 TB/s; 91 and 21.6 with one per CU, 60 and 14.7 with
// two, 49 and 13.3 with eight; 986,000: 18.8 and 5.4, 29 and 6.5, 21.5 and 5.4,
// 18.5 and 6.8)
constexpr int ORTH_B = 1024;

// chunks of the vectors for nk of them: a few hundred blocks, and not so many
// partial sums that it takes the blocks of k_orth_update long to add them up
static inline int mdot_chunks(int N, int nk) {
  const int tiles = (nk + 1 + DOT_T - 1) / DOT_T;
  return std::max(1, std::min((N + 1023) / 1024, DOT_PARTS / DOT_T / tiles));
}

// part[k * gridDim.x + chunk] = partial V[k].w (k < nk) and w.w (k = nk): w is
// read once for DOT_T vectors, whose loads are in flight together
template <typename BT>
__global__ __launch_bounds__(256) void k_mdot(int N, int nk, const BT *__restrict__ V, const BT *__restrict__ w,
                                              double *__restrict__ part) {
  __shared__ double sh[DOT_T][4];
  const int k0 = blockIdx.y * DOT_T, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const BT *v[DOT_T];
  double acc[DOT_T];
#pragma unroll
  for (int q = 0; q < DOT_T; q++) {
    v[q] = k0 + q < nk ? V + (size_t)(k0 + q) * N : w;
    acc[q] = 0.0;
  }
#pragma unroll 2
  for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256) {
    const double x = (double)w[i];
#pragma unroll
    for (int q = 0; q < DOT_T; q++) acc[q] += (double)v[q][i] * x;
  }
#pragma unroll
  for (int q = 0; q < DOT_T; q++) {
    const double t = wave_sum(acc[q]);
    if (lane == 0) sh[q][wv] = t;
  }
  __syncthreads();
  const int q = threadIdx.x;
  if (q < DOT_T && k0 + q <= nk)
    part[(size_t)(k0 + q) * gridDim.x + blockIdx.x] = (sh[q][0] + sh[q][1]) + (sh[q][2] + sh[q][3]);
}

// w -= sum_k h[k] V[k], h from k_mdot's partial sums (nc chunks); out (host
// memory) = h and w.w before; wpart[block] = partial w.w after.  LDS: nk + 1
// sums (any nk up to GM_KSPACE_MAX, 32 KB).
template <typename BT>
__global__ __launch_bounds__(256) void k_orth_update(int N, int nk, int nc, const BT *__restrict__ V,
                                                     const double *__restrict__ part, BT *__restrict__ w,
                                                     double *__restrict__ wpart, double *__restrict__ out) {
  __shared__ double sh[4];
  extern __shared__ double s_h[];
  {
    // G neighbouring threads a sum: a power of two, as many as there are for
    // nk + 1 >= 2 sums, one from 129 sums on, which then go round by 256
    int G = 128;
    while (G > 1 && 256 / G < nk + 1) G >>= 1;
    const int k = threadIdx.x / G, l = threadIdx.x & (G - 1);
    double s = 0.0;
    if (k <= nk)
      for (int c = l; c < nc; c += G) s += part[(size_t)k * nc + c];
    if (G == 128) {  // two waves each
      s = wave_sum(s);
      if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
      __syncthreads();
      if (threadIdx.x < 2) s_h[threadIdx.x] = sh[2 * threadIdx.x] + sh[2 * threadIdx.x + 1];
      __syncthreads();
    } else {
      for (int o = G >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (l == 0 && k <= nk) s_h[k] = s;
      for (int q = 256 + threadIdx.x; q <= nk; q += 256) {
        s = 0.0;
        for (int c = 0; c < nc; c++) s += part[(size_t)q * nc + c];
        s_h[q] = s;
      }
      __syncthreads();
    }
  }
  if (blockIdx.x == 0)
    for (int k = threadIdx.x; k <= nk; k += 256) out[k] = s_h[k];
  double s = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256) {
    double acc = (double)w[i];
    int k = 0;
    for (; k + DOT_T <= nk; k += DOT_T) {
      BT t[DOT_T];
#pragma unroll
      for (int q = 0; q < DOT_T; q++) t[q] = V[(size_t)(k + q) * N + i];
#pragma unroll
      for (int q = 0; q < DOT_T; q++) acc -= s_h[k + q] * (double)t[q];
    }
    for (; k < nk; k++) acc -= s_h[k] * (double)V[(size_t)k * N + i];
    const BT wn = (BT)acc;
    w[i] = wn;
    s += (double)wn * (double)wn;
  }
  const double t = block_sum(s, sh);
  if (threadIdx.x == 0) wpart[blockIdx.x] = t;
}

template <typename BT>
__global__ void k_scale_into(int N, const BT *__restrict__ w, double inv, BT *__restrict__ v) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
    v[i] = (BT)((double)w[i] * inv);
}

// v = w / |w| (v untouched when w = 0), w.w from k_orth_update's nb partial
// sums; out (host memory) = w.w
template <typename BT>
__global__ __launch_bounds__(256) void k_normalise(int N, int nb, const BT *__restrict__ w,
                                                   const double *__restrict__ wpart, BT *__restrict__ v,
                                                   double *__restrict__ out) {
  __shared__ double sh[4], s_ww;
  double p = 0.0;
  for (int c = threadIdx.x; c < nb; c += 256) p += wpart[c];
  const double t = block_sum(p, sh);
  if (threadIdx.x == 0) {
    s_ww = t;
    if (blockIdx.x == 0) *out = t;
  }
  __syncthreads();
  const double hn = sqrt(s_ww);
  if (hn == 0.0) return;
  const double inv = 1.0 / hn;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256) v[i] = (BT)((double)w[i] * inv);
}

// u = sum_k y[k] V[k]; LDS: nk coefficients
template <typename BT>
__global__ void k_combine(int N, int nk, const BT *__restrict__ V, const double *__restrict__ y,
                          BT *__restrict__ u) {
  extern __shared__ double s_h[];
  for (int k = threadIdx.x; k < nk; k += blockDim.x) s_h[k] = y[k];
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
    double acc = 0.0;
    for (int k = 0; k < nk; k++) acc += s_h[k] * (double)V[(size_t)k * N + i];
    u[i] = (BT)acc;
  }
}

// x += z (x FP64, z any), r = b - r  (r holds A x on entry), both with partial r.r
template <typename ZT>
__global__ void k_add(int N, double *__restrict__ x, const ZT *__restrict__ z) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
    x[i] += (double)z[i];
}

template <typename BT>
__global__ __launch_bounds__(RED_THREADS) void k_resid(int N, const double *__restrict__ b,
                                                       const double *__restrict__ ax,
                                                       BT *__restrict__ r,
                                                       double *__restrict__ part) {
  __shared__ double sh[RED_THREADS / 64];
  double s = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
    const double v = b[i] - ax[i];
    r[i] = (BT)v;
    s += v * v;
  }
  double t = block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

static int sum_parts(gm_ctx *c, const double *d_part, int rows, int nb, double *out) {
  GM_HIP(hipMemcpyAsync(c->h_red, d_part, (size_t)rows * nb * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  GM_HIP(hipStreamSynchronize(c->stream));
  for (int k = 0; k < rows; k++) {
    double s = 0.0;
    for (int i = 0; i < nb; i++) s += c->h_red[(size_t)k * nb + i];
    out[k] = s;
  }
  return GM_OK;
}

static constexpr int KB = 256;  // blocks of the Krylov reductions

static int ensure_krylov(gm_ctx *c, int m, int prec) {
  KrylovWork &K = c->kry;
  if (K.m >= m && K.prec == prec) return GM_OK;
  if (K.d_V) hipFree(K.d_V);
  if (K.d_w) hipFree(K.d_w);
  if (K.d_z) hipFree(K.d_z);
  if (K.d_part) hipFree(K.d_part);
  if (K.d_h) hipFree(K.d_h);
  if (K.d_V32) hipFree(K.d_V32);
  if (K.d_w32) hipFree(K.d_w32);
  if (K.d_z32) hipFree(K.d_z32);
  K = KrylovWork();
  const size_t N = c->N;
  if (prec == GM_PREC_MIXED) {
    GM_HIP(hipMalloc(&K.d_V32, (size_t)(m + 1) * N * sizeof(float)));
    GM_HIP(hipMalloc(&K.d_w32, N * sizeof(float)));
    GM_HIP(hipMalloc(&K.d_z32, 2 * N * sizeof(float)));
  } else {
    GM_HIP(hipMalloc(&K.d_V, (size_t)(m + 1) * N * sizeof(double)));
  }
  GM_HIP(hipMalloc(&K.d_w, N * sizeof(double)));
  GM_HIP(hipMalloc(&K.d_z, 2 * N * sizeof(double)));
  GM_HIP(hipMalloc(&K.d_part, (DOT_PARTS + ORTH_B) * sizeof(double)));  // of the projections, of the norms
  GM_HIP(hipMalloc(&K.d_h, (m + 2) * sizeof(double)));
  K.m = m;
  K.prec = prec;
  return GM_OK;
}

// Restarted GMRES(m), right preconditioned, classical Gram-Schmidt with a
// second pass when the first one cancels more than 1/sqrt(2) of the norm,
// convergence ||b - A x|| / ||b - A x0|| < tol (Goma's AztecOO defaults
// AZ_gmres / AZ_classic / AZ_r0, src/sl_util.c:392-960).
template <typename BT, typename VT>
static int gmres_t(gm_ctx *c, const VT *a, const double *b, double *x,
                   const gm_solver_opts *o, int *its_out, double *relres) {
  const int N = c->N, m = std::max(1, std::min(o->kspace, o->max_its));  // longest cycle
  KrylovWork &K = c->kry;
  BT *V = sizeof(BT) == 8 ? (BT *)K.d_V : (BT *)K.d_V32;
  BT *w = sizeof(BT) == 8 ? (BT *)K.d_w : (BT *)K.d_w32;
  BT *z = sizeof(BT) == 8 ? (BT *)K.d_z : (BT *)K.d_z32;
  BT *u = z + N;
  double *ax = K.d_w;  // FP64 scratch for A x (FP64 mode reuses w after use)
  double *ax2 = K.d_z + N;
  const bool pc = o->precond != GM_PC_NONE;
  std::vector<double> H((size_t)(m + 1) * m, 0.0), g(m + 1), cs(m), sn(m), y(m), h(m + 2);
  const int grid = 2048;

  auto precond = [&](const BT *in, BT *out) -> int {
    if (o->precond == GM_PC_MG) {
      if constexpr (sizeof(VT) == 8) return gm_mg_apply_d(c, (const double *)a, (const double *)in, (double *)out, o);
      else return gm_mg_apply_f(c, (const float *)a, (const double *)in, (double *)out, o);
    }
    if (o->precond == GM_PC_BAND)
      return gm_band_apply(c, sizeof(VT) == 8 ? (const double *)a : nullptr, (const double *)in, (double *)out);
    if (pc) ilu_apply<BT, BT>(c, in, out);
    else k_scale_into<BT><<<grid, 256, 0, c->stream>>>(N, in, 1.0, out);
    return GM_OK;
  };

  // w against V[0 .. j], the normalised rest in vn; the projections and w.w
  // before it in h_red, w.w after it in ww
  auto orthogonalise = [&](int j, BT *vn, double *ww) -> int {
    const int nk = j + 1, nc = mdot_chunks(N, nk), nb = std::min(ORTH_B, (N + 255) / 256);
    double *wpart = K.d_part + DOT_PARTS, *out = c->h_red;
    gm_launch(c, GM_K_MDOT, (double)(nk + 1) * N * sizeof(BT), k_mdot<BT>, dim3(nc, (nk + DOT_T) / DOT_T), dim3(256), 0,
              c->stream, N, nk, (const BT *)V, (const BT *)w, K.d_part);
    gm_launch(c, GM_K_ORTH, (double)(nk + 2) * N * sizeof(BT), k_orth_update<BT>, dim3(nb), dim3(256),
              (nk + 1) * sizeof(double), c->stream, N, nk, nc, (const BT *)V, (const double *)K.d_part, w, wpart, out);
    k_normalise<BT><<<nb, 256, 0, c->stream>>>(N, nb, w, wpart, vn, out + nk + 1);
    GM_HIP(hipGetLastError());
    GM_HIP(hipStreamSynchronize(c->stream));
    *ww = out[nk + 1];
    return GM_OK;
  };

  // r0 = b - A x
  double *axp = sizeof(BT) == 8 ? ax2 : ax;
  spmv<VT, double, double>(c, a, x, axp);
  k_resid<BT><<<KB, RED_THREADS, 0, c->stream>>>(N, b, axp, w, K.d_part);
  GM_HIP(hipGetLastError());
  double s;
  int rc = sum_parts(c, K.d_part, 1, KB, &s);
  if (rc) return rc;
  const double r0 = std::sqrt(s);
  double rn = r0;
  int its = 0;
  if (r0 == 0.0) {
    *its_out = 0;
    *relres = 0.0;
    return GM_OK;
  }
  const double eta2 = 0.5;  // (1/sqrt 2)^2
  while (its < o->max_its) {
    const double beta = rn;
    k_scale_into<BT><<<grid, 256, 0, c->stream>>>(N, w, 1.0 / beta, V);
    std::fill(g.begin(), g.end(), 0.0);
    g[0] = beta;
    int j;
    for (j = 0; j < m && its < o->max_its; j++) {
      BT *vj = V + (size_t)j * N, *vn = V + (size_t)(j + 1) * N;
      if ((rc = precond(vj, z))) return rc;
      spmv<VT, BT, BT>(c, a, z, w);
      double ww;
      if ((rc = orthogonalise(j, vn, &ww))) return rc;
      std::copy(c->h_red, c->h_red + j + 1, h.begin());
      if (ww < eta2 * c->h_red[j + 1]) {
        if ((rc = orthogonalise(j, vn, &ww))) return rc;
        for (int k = 0; k <= j; k++) h[k] += c->h_red[k];
      }
      const double hn = std::sqrt(ww);
      double *hj = H.data() + (size_t)j * (m + 1);
      for (int k = 0; k <= j; k++) hj[k] = h[k];
      hj[j + 1] = hn;
      for (int k = 0; k < j; k++) {
        const double t0 = cs[k] * hj[k] + sn[k] * hj[k + 1];
        hj[k + 1] = -sn[k] * hj[k] + cs[k] * hj[k + 1];
        hj[k] = t0;
      }
      const double den = std::sqrt(hj[j] * hj[j] + hj[j + 1] * hj[j + 1]);
      cs[j] = den == 0.0 ? 1.0 : hj[j] / den;
      sn[j] = den == 0.0 ? 0.0 : hj[j + 1] / den;
      hj[j] = den;
      hj[j + 1] = 0.0;
      g[j + 1] = -sn[j] * g[j];
      g[j] = cs[j] * g[j];
      its++;
      if (std::fabs(g[j + 1]) / r0 < o->lin_tol || hn == 0.0) {
        j++;
        break;
      }
    }
    for (int k = j - 1; k >= 0; k--) {
      double t = g[k];
      for (int l = k + 1; l < j; l++) t -= H[(size_t)l * (m + 1) + k] * y[l];
      y[k] = t / H[(size_t)k * (m + 1) + k];
    }
    GM_HIP(hipMemcpyAsync(K.d_h, y.data(), j * sizeof(double), hipMemcpyHostToDevice, c->stream));
    k_combine<BT><<<grid, 256, j * sizeof(double), c->stream>>>(N, j, V, K.d_h, u);
    if ((rc = precond(u, z))) return rc;
    k_add<BT><<<grid, 256, 0, c->stream>>>(N, x, z);
    spmv<VT, double, double>(c, a, x, axp);
    k_resid<BT><<<KB, RED_THREADS, 0, c->stream>>>(N, b, axp, w, K.d_part);
    GM_HIP(hipGetLastError());
    if ((rc = sum_parts(c, K.d_part, 1, KB, &s))) return rc;
    rn = std::sqrt(s);
    if (rn / r0 < o->lin_tol) break;
  }
  *its_out = its;
  *relres = rn / r0;
  return GM_OK;
}

// A restart cycle keeps min(kspace, max_its) vectors; a length below 1 would
// never advance.
int gm_kspace_check(const gm_solver_opts *o) {
  if (o->kspace >= 1 && std::min(o->kspace, o->max_its) <= GM_KSPACE_MAX) return GM_OK;
  gm_set_error("GMRES restart length %d outside [1, %d]", o->kspace, GM_KSPACE_MAX);
  return GM_ERR_ARG;
}

int gm_gmres_run(gm_ctx *c, const double *val, const float *val32, const double *b, double *x,
                 const gm_solver_opts *o, int *its, double *relres) {
  if (o->kspace < 1 || o->kspace > 120) {
    gm_set_error("kspace must be in [1, 120]");
    return GM_ERR_ARG;
  }
  const int prec = o->precision;
  int rc = ensure_krylov(c, o->kspace, prec);
  if (rc) return rc;
  if (o->precond == GM_PC_ILU0) {
    int bins = o->patch_bins > 0 ? o->patch_bins : gm_default_bins(c);
    if ((rc = gm_ilu_plan(c, bins))) return rc;
    if ((rc = gm_ilu_factor(c, val, val32, prec))) return rc;
  } else if (o->precond == GM_PC_BAND) {
    if ((rc = gm_band_factor(c, val, val32, prec))) return rc;
  } else if (o->precond == GM_PC_MG &&
             (!c->mg0.d_ainv || c->mg0.d_ainv != c->mg0.d_ainv_p[prec == GM_PREC_MIXED ? 1 : 0])) {
    gm_set_error("multigrid preconditioner not set up (gm_mg_setup_dev)");
    return GM_ERR_ARG;
  }
  return gm_gmres_run_nofactor(c, val, val32, b, x, o, its, relres);
}

int gm_gmres_run_nofactor(gm_ctx *c, const double *val, const float *val32, const double *b,
                          double *x, const gm_solver_opts *o, int *its, double *relres) {
  const int prec = o->precision;
  int rc = gm_kspace_check(o);
  if (rc || (rc = ensure_krylov(c, o->kspace, GM_PREC_FP64))) return rc;
  if (prec == GM_PREC_MIXED) {
    if (!val32) {
      gm_set_error("mixed precision needs FP32 Jacobian values");
      return GM_ERR_ARG;
    }
    // FP32 Jacobian values and preconditioner; Krylov basis, dot products
    // and the update in FP64
    return gmres_t<double, float>(c, val32, b, x, o, its, relres);
  }
  return gmres_t<double, double>(c, val, b, x, o, its, relres);
}

void gm_free_linalg(gm_ctx *c) {
  free_plan(c->ilu);
  KrylovWork &K = c->kry;
  void *ptrs[] = {K.d_V, K.d_w, K.d_z, K.d_part, K.d_h, K.d_V32, K.d_w32, K.d_z32};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  c->kry = KrylovWork();
}

int gm_ilu_factor_export(gm_ctx *c, const double *val, int bins, int *rowptr, int *col, double *lu) {
  int rc = gm_ilu_plan(c, bins);
  if (rc) return rc;
  if ((rc = gm_ilu_factor(c, val, nullptr, GM_PREC_FP64))) return rc;
  IluPlan &P = c->ilu;
  GM_HIP(hipMemcpy(rowptr, P.d_rowptr, (c->N + 1) * sizeof(int), hipMemcpyDeviceToHost));
  GM_HIP(hipMemcpy(col, P.d_col, P.nnz * sizeof(int), hipMemcpyDeviceToHost));
  GM_HIP(hipMemcpy(lu, P.d_lu, P.nnz * sizeof(double), hipMemcpyDeviceToHost));
  return (int)P.nnz;
}
