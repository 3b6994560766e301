// Geometric multigrid preconditioner with element-block (Vanka) smoothing.
//
// Levels: level 0 is the context's own mesh and (row-sum-scaled) Jacobian;
// coarser levels are contexts on coarsened meshes whose Jacobians are
// re-assembled by the same fill kernels at the injected state.  Transfers are
// CSR matrices P (coarse -> fine) and R = P^T supplied by the caller.
//
// Smoother: for each element colour, r = b - A x on every row, then every
// element of the colour solves its local system (all velocity, temperature
// and pressure unknowns of the element, entries taken from the assembled
// matrix through the element-to-nonzero map) and adds omega * A_e^-1 r_e to x.
// Elements of one colour share no unknowns, and the residual is formed before
// the colour's updates, so the sweep is deterministic (block Gauss-Seidel
// across colours, block Jacobi within a colour).  The local inverses are
// formed once per Newton step by Gauss-Jordan elimination with partial
// pivoting in registers.
#include <algorithm>
#include <cmath>
#include <vector>

#include "gm_launch.h"

template <int DIM, int EN>
struct Loc {
  static constexpr int NVE = DIM == 2 ? 9 : 27;
  static constexpr int NP = DIM + 1;
  static constexpr int NV = DIM + EN;
  static constexpr int N = NV * NVE + NP;
};

struct LevelDev {
  const int *conn, *fu, *centroid, *e2nz, *bindx;
  const signed char *dbc;
  long long E, off_mp, off_cv, off_cp;
};

template <int DIM, int EN>
__device__ inline int local_dof(const LevelDev &L, int e, int li) {
  using Lc = Loc<DIM, EN>;
  if (li < Lc::NV * Lc::NVE) {
    const int a = li / Lc::NVE, i = li - a * Lc::NVE;
    return L.fu[L.conn[(size_t)e * Lc::NVE + i]] + a;
  }
  return L.fu[L.centroid[e]] + DIM + EN + (li - Lc::NV * Lc::NVE);
}

// e2nz position of local entry (li, lj), -1 when the pair is not in the graph
template <int DIM, int EN>
__device__ inline long long local_pos(const LevelDev &L, int li, int lj) {
  using Lc = Loc<DIM, EN>;
  constexpr int NVE = Lc::NVE, NP = Lc::NP, NV = Lc::NV, NN = NV * NVE;
  if (li < NN) {
    const int a = li / NVE, i = li - a * NVE;
    if (lj < NN) {
      const int b = lj / NVE, j = lj - b * NVE;
      return (long long)(a * NV + b) * NVE * NVE + i * NVE + j;
    }
    if (a >= DIM) return -1;  // energy row x pressure column: not in the graph
    return L.off_mp + (long long)a * NVE * NP + i * NP + (lj - NN);
  }
  const int k = li - NN;
  if (lj < NN) {
    const int b = lj / NVE, j = lj - b * NVE;
    if (b >= DIM) return -1;  // continuity x temperature: identically zero
    return L.off_cv + (long long)b * NP * NVE + k * NVE + j;
  }
  return L.off_cp + (long long)k * NP + (lj - NN);
}

// The pivot's rank of |v|, all of its bits: 0 for a used row, 1 for a zero or a
// NaN, else the bits + 2, which order as the values do
__device__ inline unsigned long long pivot_rank(double v, bool used) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v) & ~(1ull << 63);
  return used ? 0ull : fabs(v) > 0.0 ? b + 2ull : 1ull;
}
__device__ inline unsigned pivot_rank(float v, bool used) {
  return used ? 0u : fabsf(v) > 0.0f ? (__builtin_bit_cast(unsigned, v) & 0x7fffffffu) + 2u : 1u;
}
// v of lane i (the same i in every lane)
__device__ inline unsigned rank_of(unsigned v, int i) { return (unsigned)__builtin_amdgcn_readlane((int)v, i); }
__device__ inline unsigned long long rank_of(unsigned long long v, int i) {
  return (unsigned long long)rank_of((unsigned)(v >> 32), i) << 32 | rank_of((unsigned)v, i);
}

// local matrix -> inverse (stored transposed: ainv[e][j][i] = (A_e^-1)[i][j])
// QUAD9 element blocks (at most 32 unknowns) by Gauss-Jordan with partial
// pivoting in compute type CT (FP64, or FP32 for the mixed precision), two
// blocks per wave: lane i of a half holds row i in registers.  Rows stay
// where they are; step k takes the unused row with the largest entry of
// column k (the first on ties), which passes through LDS within the wave: two
// reads a lane, then DPP broadcasts.  The pivot row waits for its scale until it
// is stored.  No workgroup barrier.  A structurally empty column (a local
// pressure mode with no velocity coupling inside the element) leaves that
// unknown untouched.
// Measured (16384 blocks of 30 unknowns, FP64): 186 us against 450 with a
// workgroup per block in LDS and three barriers a step.
template <int DIM, int EN, typename VT, typename AT, typename CT>
__global__ __launch_bounds__(256) void k_vanka_invert(LevelDev L, int nelem, const VT *__restrict__ val,
                                                      AT *__restrict__ ainv) {
  using Lc = Loc<DIM, EN>;
  constexpr int n = Lc::N;
  static_assert(n <= 32, "a row per lane of half a wave");
  __shared__ CT s_row[8][32], s_turn[8][8][33];
  __shared__ int s_piv[8][32];
  const int lane = threadIdx.x & 63, sub = threadIdx.x >> 5, i = lane & 31, l16 = lane & 15;
  const int e = blockIdx.x * 8 + sub;
  const bool act = e < nelem && i < n;
  const int *map = L.e2nz + (size_t)(act ? e : 0) * L.E;
  CT P[n] = {};
  CT scale = 0;
  bool used = i >= n;
  int st = 0;
  // eight rows at a time, a lane per column (neighbouring columns are mostly
  // neighbours in memory), turned through LDS to a lane per row
#pragma unroll
  for (int r0 = 0; r0 < n; r0 += 8) {
    CT v[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const long long p = act && r0 + r < n ? local_pos<DIM, EN>(L, r0 + r, i) : -1;
      v[r] = p >= 0 ? (CT)val[map[p]] : (CT)0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < 8; r++) s_turn[sub][r][i] = v[r];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (i >= r0 && i < r0 + 8)
#pragma unroll
      for (int j = 0; j < n; j++) P[j] = s_turn[sub][i - r0][j];
  }
  // the columns move up one register a step, so that the step's is the first
#pragma unroll 1
  for (int k = 0; k < n; k++) {
    const auto key = pivot_rank(P[0], used), m = row_max16(key);
    const auto a = rank_of(m, 0), b = rank_of(m, 16), c = rank_of(m, 32), d = rank_of(m, 48);
    const unsigned long long at = __ballot(key == (lane < 32 ? max(a, b) : max(c, d)));
    const int p = __ffs(lane < 32 ? (unsigned)at : (unsigned)(at >> 32)) - 1;
    const bool is = i == p;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (is) {
#pragma unroll
      for (int j = 0; j < n; j++) s_row[sub][j] = P[j];
      s_piv[sub][k] = p;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const CT lo = s_row[sub][l16], hi = s_row[sub][16 + l16];
    const CT piv = row_bcast(lo, 0);
    const CT dv = fabs(piv) > (CT)1e-300 ? reciprocal(piv) : (CT)0;
    // the pivot row waits for its scale dv until it is stored
    const CT f = is ? (CT)0 : P[0] * dv;
    used = used || is;
    st = is ? k : st;
    scale = is ? dv : scale;
#pragma unroll
    for (int j = 1; j < n; j++) {
      P[j - 1] = fma(row_bcast(j < 16 ? lo : hi, j & 15), -f, P[j]);
      if (j % 8 == 0) __builtin_amdgcn_sched_barrier(0);  // eight broadcasts ahead, not all: no spills
    }
    P[n - 1] = is ? (CT)1 : -f;
  }
  if (!act) return;
  // row i is inverse row st; its column c belongs to the pivot row of step c
  AT *out = ainv + (size_t)e * n * n + st;
#pragma unroll
  for (int c = 0; c < n; c++) out[s_piv[sub][c] * n] = (AT)(scale * P[c]);
}

// the larger |entry| of (best, bi) and the lane R places along; lower row on ties
template <int R, typename CT>
__device__ inline void pivot_combine(CT &best, int &bi) {
  const CT ov = row_ror_f<R>(best);
  const int oi = row_ror_i<R>(bi);
  if (ov > best || (ov == best && oi < bi)) {
    best = ov;
    bi = oi;
  }
}

// Pivot of one column: the TR lanes of one DPP row hold its entries cv[a]
// (rows tr + TR a).  They stage the column in col, pick the row not yet used
// (bit a of `used`) with the largest |entry| (a NaN counts as zero, ties go to
// the lower row, so an unused row is always found), and the lane holding it
// posts the row to *pp, its reciprocal to *dv (0 for a structurally empty
// column: a local pressure mode with no velocity coupling inside the element,
// which leaves that unknown untouched) and clears the row's factor in col.
template <int n, int RA, int TR, typename CT>
__device__ inline void post_pivot(const CT (&cv)[RA], unsigned used, int tr, CT *col, int *pp,
                                  CT *dv) {
  CT best = (CT)-1;
  int bi = n;
#pragma unroll
  for (int a = 0; a < RA; a++) {
    const int i = tr + TR * a;
    const CT v = cv[a];
    col[i] = v;
    CT m = fabs(v);
    m = m == m ? m : (CT)0;
    if ((n % TR == 0 || i < n) && !((used >> a) & 1u) && m > best) {
      best = m;
      bi = i;
    }
  }
  pivot_combine<8>(best, bi);
  pivot_combine<4>(best, bi);
  pivot_combine<2>(best, bi);
  pivot_combine<1>(best, bi);
  if (tr == (bi & (TR - 1))) {
    const CT pv = col[bi];
    *dv = fabs(pv) > (CT)1e-300 ? (CT)1 / pv : (CT)0;
    col[bi] = (CT)0;
    *pp = bi;
  }
}

// The same inverse with the block held in registers: thread (tr, tc) of a
// TR x TC grid owns rows tr + TR a and columns tc + TC b.  Pivoting is
// implicit: step k takes its pivot row p_k among the rows not yet used and
// leaves every row where it is.  Scaling is lazy: the pivot row keeps its
// entries (column k set to 1) and is multiplied by its pivot's reciprocal d_k
// when the block is written out; the other rows subtract f (d_k row) as usual.
// The stored result M then holds the inverse with both permutations applied,
// inv[k][p_c] = d_k M[p_k][c], undone at the write.  So no register is
// written under a runtime row index: the loop over column blocks is unrolled
// (column k's registers are addressed at compile time) and the pivot row is
// read through a scalar switch on its block index, which is uniform over the
// workgroup.  One barrier a step: the lanes owning column k post its pivot,
// the pivot's reciprocal and the column in LDS (double-buffered by step
// parity); the pivot row's entries that a thread needs are held by lanes of
// its own wave (row rp, same tc) and pass through LDS within the wave.
template <int DIM, int EN, typename VT, typename AT, typename CT, int TR, int TC>
__global__ __launch_bounds__(TR *TC) void k_vanka_invert_reg(LevelDev L, const VT *__restrict__ val,
                                                             AT *__restrict__ ainv) {
  using Lc = Loc<DIM, EN>;
  constexpr int n = Lc::N;
  constexpr int RA = (n + TR - 1) / TR, CB = (n + TC - 1) / TC;
  static_assert(RA <= 8, "pivot-row switch covers eight row blocks");
  static_assert(TR == 16, "a column's TR lanes form one DPP row");
  // every row / column index of the thread grid is inside the block
  constexpr bool RFULL = n % TR == 0, CFULL = n % TC == 0;
  __shared__ CT s_col[2][RA * TR], s_row[CB * TC], s_dv[2], s_d[n];
  __shared__ int s_prow[n], s_kinv[n], s_pp[2];
  const int e = blockIdx.x, tid = threadIdx.x;
  const int tr = tid % TR, tc = tid / TR;
  const int *map = L.e2nz + (size_t)e * L.E;
  CT A[RA][CB];
#pragma unroll
  for (int a = 0; a < RA; a++)
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const int i = tr + TR * a, j = tc + TC * b;
      const long long p = ((RFULL || i < n) && (CFULL || j < n)) ? local_pos<DIM, EN>(L, i, j) : -1;
      A[a][b] = p >= 0 ? (CT)val[map[p]] : (CT)0;
    }
  unsigned used = 0;  // bit a: row tr + TR a has been a pivot row
#pragma unroll
  for (int K = 0; K < CB; K++) {
    for (int r = 0; r < TC; r++) {
      const int k = TC * K + r;
      if (k >= n) break;
      const int q = k & 1;
      if (tc == r) {
        CT cv[RA];
#pragma unroll
        for (int a = 0; a < RA; a++) cv[a] = A[a][K];
        post_pivot<n, RA, TR>(cv, used, tr, s_col[q], &s_pp[q], &s_dv[q]);
      }
      __syncthreads();
      const int p = __builtin_amdgcn_readfirstlane(s_pp[q]);
      const CT d = s_dv[q];
      if (tid == 0) {
        s_prow[k] = p;
        s_kinv[p] = k;
        s_d[k] = d;
      }
      const int ap = p / TR, rp = p - ap * TR;
      // This wave's columns of the pivot row pass through s_row: the lanes of
      // row p write them and the same wave reads them back (LDS keeps one
      // wave's operations in order; the fences keep the compiler from moving
      // the reads above the writes), so no workgroup barrier is needed.
      if (tr == rp) {
        switch (ap) {
#define GM_PIVOT_ROW(c)                                            \
  case c:                                                          \
    if constexpr (c < RA) {                                        \
      _Pragma("unroll") for (int b = 0; b < CB; b++) {             \
        const int j = tc + TC * b;                                 \
        if (CFULL || j < n) s_row[j] = A[c][b];                    \
      }                                                            \
    }                                                              \
    break;
          GM_PIVOT_ROW(0) GM_PIVOT_ROW(1) GM_PIVOT_ROW(2) GM_PIVOT_ROW(3)
          GM_PIVOT_ROW(4) GM_PIVOT_ROW(5) GM_PIVOT_ROW(6) GM_PIVOT_ROW(7)
#undef GM_PIVOT_ROW
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // Step k of Gauss-Jordan on pivot row p: every other row i subtracts f_i
      // times d row p (f_i its column-k entry) and takes -f_i d in column k;
      // row p keeps its entries, with 1 in column k.  One FMA per entry after
      // column k is set to 1 (row p) and 0 (the others); f_p is 0.
      CT rb[CB], fa[RA];
#pragma unroll
      for (int b = 0; b < CB; b++) {
        const int j = tc + TC * b;
        rb[b] = (CFULL || j < n) ? s_row[j] * d : (CT)0;
      }
      rb[K] = tc == r ? d : rb[K];
#pragma unroll
      for (int a = 0; a < RA; a++) fa[a] = s_col[q][tr + TR * a];
      if (tc == r) {
#pragma unroll
        for (int a = 0; a < RA; a++) A[a][K] = tr + TR * a == p ? (CT)1 : (CT)0;
      }
#pragma unroll
      for (int a = 0; a < RA; a++)
#pragma unroll
        for (int b = 0; b < CB; b++) A[a][b] -= fa[a] * rb[b];
      if (tr == rp) used |= 1u << ap;
    }
  }
  __syncthreads();
  AT *out = ainv + (size_t)e * n * n;
#pragma unroll
  for (int a = 0; a < RA; a++) {
    const int i = tr + TR * a;
    if (!RFULL && i >= n) continue;
    const int ki = s_kinv[i];
    const CT di = s_d[ki];
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const int c = tc + TC * b;
      if (CFULL || c < n) out[(size_t)s_prow[c] * n + ki] = (AT)(A[a][b] * di);
    }
  }
}

// r = b - A x over all rows (MSR), G lanes per row
template <typename VT, typename BT, int G>
__global__ __launch_bounds__(256) void k_mg_resid(int N, const VT *__restrict__ a,
                                                  const int *__restrict__ bindx,
                                                  const BT *__restrict__ x,
                                                  const BT *__restrict__ b, BT *__restrict__ r) {
  const int row = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (row >= N) return;
  using AT = typename std::conditional<sizeof(BT) == 8, double, float>::type;
  const int k0 = bindx[row], k1 = bindx[row + 1];
  AT s = row_dot<AT, VT, BT, G>(a, bindx, x, k0, k1, lane);
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (lane == 0) r[row] = (BT)((AT)b[row] - s - (AT)a[row] * (AT)x[row]);
}

// r = b - A x on a list of rows (the unknowns of one element colour)
template <typename VT, typename BT, int G>
__global__ __launch_bounds__(256) void k_mg_resid_rows(int nrows, const int *__restrict__ rows,
                                                       const VT *__restrict__ a,
                                                       const int *__restrict__ bindx,
                                                       const BT *__restrict__ x,
                                                       const BT *__restrict__ b, BT *__restrict__ r) {
  const int k = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (k >= nrows) return;
  const int row = rows[k];
  using AT = typename std::conditional<sizeof(BT) == 8, double, float>::type;
  const int k0 = bindx[row], k1 = bindx[row + 1];
  AT s = row_dot<AT, VT, BT, G>(a, bindx, x, k0, k1, lane);
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (lane == 0) r[row] = (BT)((AT)b[row] - s - (AT)a[row] * (AT)x[row]);
}

// ---- exact coarse solve: dense inverse by Gauss-Jordan with partial
// pivoting, applied as a dense GEMV.

template <typename VT>
__global__ void k_msr_to_dense(int n, const VT *__restrict__ a, const int *__restrict__ bindx,
                               double *__restrict__ D) {
  const int row = blockIdx.x;
  for (int k = bindx[row] + threadIdx.x; k < bindx[row + 1]; k += blockDim.x)
    D[(size_t)row * n + bindx[k]] = (double)a[k];
  if (threadIdx.x == 0) D[(size_t)row * n + row] = (double)a[row];
}

// Dense Gauss-Jordan inverse of the coarsest level with partial pivoting,
// blocked in panels of NB columns.  Rows stay where they are: step k takes as
// pivot the unused row with the largest entry of column k (the first on ties),
// and the finished array holds inverse row k in the row that
// was step k's pivot, its columns in pivot order too (k_gj_permute).
//
// One launch per panel, from one copy D of the array into the other, O:
//   the tiles apply panel K to the other columns, O = D' + Pan D_K: Pan the
//     panel's columns after its steps, D_K its pivot rows, D' = D with those
//     rows zeroed; panel K's own columns become Pan;
//   the first workgroup meanwhile brings panel K + 1 up to date in registers
//     and runs its column steps.
// A panel's terms of an entry are added up from zero and to the entry once:
// added one by one they left 1.6 times the residual (1059 unknowns).
// The panel workgroup is a chain of dependent steps that the tiles hide behind
// (for 1480 unknowns they take 17 us of the launch): thread t owns rows
// t + NT r of the panel.  Per step each group of 16 lanes finds its candidate
// with two 32-bit maxima (DPP rotations); the lane that holds it puts its key,
// its reciprocal and its row into LDS, and after the step's only barrier every
// wave picks the winner.  The buffers alternate by step parity, so no second
// barrier guards their reuse.  Few waves with several rows a thread: the step
// is latency, not work.
// Measured: 33 us a panel of 16 for 1480 unknowns, 22 for 532, 14 for 87,
// against 80, 59 and 46 with row interchanges, two barriers a step and launches
// of their own for the panel, the interchanges and the update; the rows'
// final order costs 9 us instead of 295.
constexpr int GJ_NB = 16;  // widest panel

template <int NB, int RPT, int NT>
__global__ __launch_bounds__(NT) void k_gjb_step(int n, int kb, int nb, int kb2, int nb2,
                                                 const double *__restrict__ D, double *__restrict__ O,
                                                 const double *__restrict__ pan, double *__restrict__ pan2,
                                                 const int *__restrict__ piv, int *__restrict__ piv2,
                                                 int *stepof, int *__restrict__ flag) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, lq = lane >> 4;
  constexpr int NW = NT / 64;
  typedef double d4 __attribute__((ext_vector_type(4)));
  if (blockIdx.x == 0) {
    if (nb2 == 0) return;
    constexpr int NG = 4 * NW, NK = NG / 16;  // groups of 16 lanes, keys per lane
    struct Cand {
      double v[4], inv;
      int row;
    };
    __shared__ Cand s_cand[2][NG];
    __shared__ unsigned long long s_key[2][NG];
    __shared__ double s_old[4][NB - 4];
    __shared__ double s_turn[NW][16][17];
    // panel K + 1's columns with panel K applied, 16 rows at a time on the
    // matrix cores (as the tiles below), turned through LDS to a row per thread
    // rows loaded together and sets of 16 lanes of them, as registers allow
    constexpr int RB = NT == 256 ? RPT : 1, MB = NT == 1024 ? 2 : 4;
    double P[RPT][NB], bk[NB / 4];
    bool used[RPT];
#pragma unroll
    for (int k = 0; k < NB / 4; k++) {
      const int t = 4 * k + lq;
      bk[k] = t < nb ? D[(size_t)piv[t] * n + kb2 + l16] : 0.0;
    }
    unsigned long long zero[RPT];  // rows that start from zero: the pivot rows of panel K
#pragma unroll
    for (int r = 0; r < RPT; r++) {
      const int i = NT * r + tid, at = i < n && kb2 > 0 ? stepof[i] : -1;
      used[r] = i >= n || at >= 0;
      zero[r] = __ballot(i >= n || (nb > 0 && at >= kb && at < kb + nb));
    }
#pragma unroll
    for (int r0 = 0; r0 < RPT; r0 += RB)
#pragma unroll
      for (int m0 = 0; m0 < 4; m0 += MB) {
        d4 B[RB][MB], C[RB][MB];  // the columns before, what panel K adds
        double f[RB][MB][NB / 4];
#pragma unroll
        for (int r = 0; r < RB; r++) {
          const int ib = NT * (r0 + r) + 64 * w + 16 * m0;
#pragma unroll
          for (int m = 0; m < MB; m++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const int row = 16 * m + lq + 4 * e;
              // past the last column: another row's, or the margin; unused
              B[r][m][e] = (zero[r0 + r] >> (16 * m0 + row)) & 1 ? 0.0 : D[(size_t)(ib + row) * n + kb2 + l16];
            }
            C[r][m] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < NB / 4; k++) {
              const int t = 4 * k + lq;
              f[r][m][k] = t < nb && ib + 16 * m + l16 < n ? pan[(size_t)t * n + ib + 16 * m + l16] : 0.0;
            }
          }
        }
        if (nb > 0)
#pragma unroll
          for (int k = 0; k < NB / 4; k++)
#pragma unroll
            for (int r = 0; r < RB; r++)
#pragma unroll
              for (int m = 0; m < MB; m++)
                C[r][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[r][m][k], bk[k], C[r][m], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
          for (int m = 0; m < MB; m++) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int e = 0; e < 4; e++) s_turn[w][lq + 4 * e][l16] = B[r][m][e] + C[r][m][e];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (lq == m0 + m)
#pragma unroll
              for (int j = 0; j < NB; j++) P[r0 + r][j] = s_turn[w][l16][j];
          }
      }
    int step[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) step[r] = -1;
    __syncthreads();
    // Four columns at a time, the others brought up to date after the four: a
    // step then waits for four values of its pivot row, not for sixteen.  The
    // columns move up four registers a round, so that the round's are always
    // the first and the loop stays in the instruction cache.
#pragma unroll 1
    for (int c0 = 0; c0 < nb2; c0 += 4) {
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        if (c0 + kk >= nb2) continue;
        const int q = kk & 1;
        unsigned long long best = 0;  // pivot_rank of the thread's candidate
        int br = 0;
        double cand[4] = {P[0][0], P[0][1], P[0][2], P[0][3]};
#pragma unroll
        for (int r = 0; r < RPT; r++) {
          const unsigned long long key = pivot_rank(P[r][kk], used[r]);
          if (r == 0 || key > best) {
            best = key;
            br = r;
#pragma unroll
            for (int j = 0; j < 4; j++) cand[j] = P[r][j];
          }
        }
        double ci = reciprocal(cand[kk]);  // every lane's, beside the chain of the maximum
        asm volatile("" : "+v"(ci));
        const unsigned long long m = row_max16(best), at = __ballot(best == m);
        if (lane == 16 * lq + __ffs((unsigned)(at >> (16 * lq)) & 0xffffu) - 1) {  // the first of its 16 lanes
          Cand &c = s_cand[q][4 * w + lq];
          s_key[q][4 * w + lq] = m;
          c.row = tid + NT * br;
          c.inv = ci;
#pragma unroll
          for (int j = 0; j < 4; j++) c.v[j] = cand[j];
        }
        __syncthreads();
        unsigned long long wk[NK], wm = 0;
#pragma unroll
        for (int c = 0; c < NK; c++) {
          wk[c] = s_key[q][NK * l16 + c];
          wm = max(wm, wk[c]);
        }
        wm = row_max16(wm);
        int g = 0;  // a group that has the maximum, the same in every wave
#pragma unroll
        for (int c = NK - 1; c >= 0; c--) {
          const unsigned long long has = __ballot(wk[c] == wm);
          g = has ? NK * (__ffsll(has) - 1) + c : g;
        }
        const Cand &c = s_cand[q][__builtin_amdgcn_readfirstlane(g)];
        const double inv = c.inv, R[4] = {c.v[0], c.v[1], c.v[2], c.v[3]};
        const int p = __builtin_amdgcn_readfirstlane(c.row);
        if (tid == 0) {
          piv2[c0 + kk] = p;
          if (wm == 1) flag[3] = 1;  // singular coarse matrix
        }
#pragma unroll
        for (int r = 0; r < RPT; r++) {
          const bool is = p == tid + NT * r;  // the pivot row: R inv, and inv itself
          const double f = is ? -inv : P[r][kk] * inv;
          used[r] = used[r] || is;
          step[r] = is ? kb2 + c0 + kk : step[r];
#pragma unroll
          for (int j = 0; j < 4; j++) P[r][j] = j == kk ? -f : fma(R[j], -f, is ? 0.0 : P[r][j]);
        }
      }
      // the other columns: zero in the four pivot rows, plus the four columns
      // times those rows' old values
#pragma unroll
      for (int r = 0; r < RPT; r++)
        if (step[r] >= kb2 + c0) {
          double *old = s_old[step[r] - kb2 - c0];
#pragma unroll
          for (int j = 4; j < NB; j++) {
            old[j - 4] = P[r][j];
            P[r][j] = 0.0;
          }
        }
      __syncthreads();
      double mine[4];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) mine[kk] = s_old[kk][l16 < NB - 4 ? l16 : 0];
      double Q[RPT][NB];
#pragma unroll
      for (int r = 0; r < RPT; r++)
#pragma unroll
        for (int j = 4; j < NB; j++) Q[r][j - 4] = P[r][j];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        if (c0 + kk >= nb2) continue;
        double R[NB - 4];
#pragma unroll
        for (int j = 0; j < NB - 4; j++) R[j] = row_bcast(mine[kk], j);
        __builtin_amdgcn_sched_barrier(0);  // the moves together, not each waited for by its products
#pragma unroll
        for (int j = 0; j < NB - 4; j++)
#pragma unroll
          for (int r = 0; r < RPT; r++) Q[r][j] = fma(R[j], P[r][kk], Q[r][j]);
      }
#pragma unroll
      for (int r = 0; r < RPT; r++) {
#pragma unroll
        for (int j = 0; j < 4; j++) Q[r][NB - 4 + j] = P[r][j];
#pragma unroll
        for (int j = 0; j < NB; j++) P[r][j] = Q[r][j];
      }
    }
    const int moved = (nb2 + 3) & ~3;
#pragma unroll
    for (int r = 0; r < RPT; r++) {
      const int i = tid + NT * r;
      if (i >= n) continue;
      if (step[r] >= 0 || kb2 == 0) stepof[i] = step[r];
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const int c = (j + moved) & (NB - 1);  // the column here by now
        if (c < nb2) pan2[(size_t)c * n + i] = P[r][j];
      }
    }
    return;
  }
  // 16 x 64 tiles, one per wave, on the matrix cores: lane l supplies
  // A[l%16][l/16] and B[l/16][l%16] and holds D[l/16 + 4r][l%16]
  const int tx = (n + 63) / 64, task = ((int)blockIdx.x - 1) * NW + w;
  const int i0 = task / tx * 16, j0 = (task - task / tx * tx) * 64;
  if (i0 >= n) return;
  d4 B[4], C[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int i = i0 + lq + 4 * r;
    const int at = i < n ? stepof[i] : -1;
    const bool zero = i >= n || (at >= kb && at < kb + nb);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int j = j0 + 16 * c + l16;
      B[c][r] = zero || j >= n ? 0.0 : D[(size_t)i * n + j];
      C[c][r] = 0.0;
    }
  }
#pragma unroll
  for (int k = 0; k < NB; k += 4) {
    const int t = k + lq;
    const double a = t < nb && i0 + l16 < n ? pan[(size_t)t * n + i0 + l16] : 0.0;
    const double *row = D + (size_t)(t < nb ? piv[t] : 0) * n;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int j = j0 + 16 * c + l16;
      const double d = t < nb && j < n ? row[j] : 0.0;
      C[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, d, C[c], 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int i = i0 + lq + 4 * r;
    if (i >= n) continue;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int j = j0 + 16 * c + l16;
      if (j >= n || (j >= kb2 && j < kb2 + nb2)) continue;  // the next launch writes panel K + 1
      O[(size_t)i * n + j] = j >= kb && j < kb + nb ? pan[(size_t)(j - kb) * n + i] : B[c][r] + C[c][r];
    }
  }
}

// inverse[k][c] = D[pivot of k][step of c]
__global__ __launch_bounds__(256) void k_gj_permute(int n, const int *__restrict__ piv, const int *__restrict__ stepof,
                                                    const double *__restrict__ D, double *__restrict__ G) {
  const int k = blockIdx.x;
  const double *row = D + (size_t)piv[k] * n;
  for (int c = threadIdx.x; c < n; c += 256) G[(size_t)k * n + c] = row[stepof[c]];
}

// x = D b, one wave per row
template <typename BT>
__global__ __launch_bounds__(256) void k_dense_gemv(int n, const double *__restrict__ D,
                                                    const BT *__restrict__ b, BT *__restrict__ x) {
  const int row = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (row >= n) return;
  const double *r = D + (size_t)row * n;
  double s = 0.0;
  for (int j = lane; j < n; j += 64) s += r[j] * (double)b[j];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) x[row] = (BT)s;
}

// x_e += omega * A_e^-1 r_e for the nelem elements of one colour
template <int DIM, int EN, typename AT, typename BT, int NT>
__global__ __launch_bounds__(NT) void k_vanka_update(LevelDev L, int nelem, const int *__restrict__ elems,
                                                     const AT *__restrict__ ainv,
                                                     const BT *__restrict__ r, BT *__restrict__ x,
                                                     double omega, const double *__restrict__ wmul) {
  using Lc = Loc<DIM, EN>;
  constexpr int n = Lc::N;
  // two elements per workgroup when a block fits in half of it (2D: 30 of 64 lanes)
  constexpr int EPB = (2 * n <= NT) ? 2 : 1;
  constexpr int HALF = NT / EPB;
  __shared__ double s_r2[EPB][n];
  __shared__ int s_g2[EPB][n];
  const int tid = threadIdx.x, sub = tid / HALF, t = tid - sub * HALF;
  const int eidx = xcd_block() * EPB + sub;
  const bool act = eidx < nelem;
  const int e = act ? elems[eidx] : 0;
  if (act)
    for (int i = t; i < n; i += HALF) {
      const int g = local_dof<DIM, EN>(L, e, i);
      s_g2[sub][i] = g;
      s_r2[sub][i] = (double)r[g];
    }
  __syncthreads();
  if (act) {
    const AT *M = ainv + (size_t)e * n * n;
    for (int i = t; i < n; i += HALF) {
      double s = 0.0;
      for (int j = 0; j < n; j++) s += (double)M[j * n + i] * s_r2[sub][j];
      const int g = s_g2[sub][i];
      x[g] += (BT)(omega * (wmul ? wmul[g] : 1.0) * s);
    }
  }
}

// Additive smoother, first half: every element's correction c_e = A_e^-1 r_e
// (all elements in one launch; nothing is written to x).
template <int DIM, int EN, typename AT, typename BT, int NT>
__global__ __launch_bounds__(NT) void k_vanka_corr(LevelDev L, int nelem, const AT *__restrict__ ainv,
                                                   const BT *__restrict__ r, double *__restrict__ corr) {
  using Lc = Loc<DIM, EN>;
  constexpr int n = Lc::N;
  constexpr int EPB = (2 * n <= NT) ? 2 : 1;
  constexpr int HALF = NT / EPB;
  __shared__ double s_r2[EPB][n];
  const int tid = threadIdx.x, sub = tid / HALF, t = tid - sub * HALF;
  const int e = xcd_block() * EPB + sub;
  const bool act = e < nelem;
  if (act)
    for (int i = t; i < n; i += HALF) s_r2[sub][i] = (double)r[local_dof<DIM, EN>(L, e, i)];
  __syncthreads();
  if (act) {
    const AT *M = ainv + (size_t)e * n * n;
    for (int i = t; i < n; i += HALF) {
      double s = 0.0;
      for (int j = 0; j < n; j++) s += (double)M[j * n + i] * s_r2[sub][j];
      corr[(size_t)e * n + i] = s;
    }
  }
}

// Second half: x_u += omega / (elements sharing u) * sum of u's corrections, in
// a fixed order (deterministic); assign: x_u = that (x is zero on entry).
template <typename BT>
__global__ __launch_bounds__(256) void k_vanka_gather(int N, const int *__restrict__ gptr,
                                                      const int *__restrict__ gent,
                                                      const double *__restrict__ corr,
                                                      const double *__restrict__ wmul, double omega,
                                                      BT *__restrict__ x, int assign) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= N) return;
  double s = 0.0;
  for (int k = gptr[u]; k < gptr[u + 1]; k++) s += corr[gent[k]];
  const BT d = (BT)(omega * wmul[u] * s);
  x[u] = assign ? d : x[u] + d;
}

// y = M v (CSR), optionally scaling v by sc and masking Dirichlet rows; G
// lanes per row (consecutive lanes read consecutive entries of the row)
template <typename BT, int G>
__global__ __launch_bounds__(256) void k_csr_apply(int nrows, const int *__restrict__ rp,
                                                   const int *__restrict__ ci,
                                                   const double *__restrict__ cv,
                                                   const BT *__restrict__ v,
                                                   const double *__restrict__ sc,
                                                   const signed char *__restrict__ mask,
                                                   BT *__restrict__ y, int accumulate) {
  const int i = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (i >= nrows) return;  // whole groups of G lanes leave together
  double s = 0.0;
  for (int k = rp[i] + lane; k < rp[i + 1]; k += G) {
    const int j = ci[k];
    s += cv[k] * (double)v[j] * (sc ? sc[j] : 1.0);
  }
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (lane) return;
  if (mask && mask[i]) s = 0.0;
  if (accumulate) y[i] += (BT)s;
  else y[i] = (BT)s;
}

// coarse state: nodal values injected from the finer level, pressure 0
__global__ void k_inject(int ncn, const int *__restrict__ inj, const int *__restrict__ fu_f,
                         const int *__restrict__ fu_c, int nv, const double *__restrict__ xf,
                         double *__restrict__ xc) {
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < ncn; n += gridDim.x * blockDim.x) {
    const int f = fu_f[inj[n]], cc = fu_c[n], cnt = fu_c[n + 1] - cc;
    for (int a = 0; a < cnt; a++) xc[cc + a] = a < nv ? xf[f + a] : 0.0;
  }
}

template <typename T>
__global__ void k_set(T *p, long long n, T v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---------------------------------------------------------------- host side

static LevelDev level_dev(const gm_ctx *c) {
  LevelDev L;
  L.conn = c->d_conn;
  L.fu = c->d_fu;
  L.centroid = c->d_centroid;
  L.e2nz = c->d_e2nz;
  L.bindx = c->d_bindx;
  L.dbc = c->d_dbc;
  L.E = c->lay.total;
  L.off_mp = c->lay.off_mp;
  L.off_cv = c->lay.off_cv;
  L.off_cp = c->lay.off_cp;
  return L;
}

static int nloc_of(const gm_ctx *c) { return c->nv * c->nve + c->np; }

template <typename T>
static int upv(T **d, const T *h, size_t n) {
  GM_HIP(hipMalloc(d, std::max<size_t>(n, 1) * sizeof(T)));
  if (n) GM_HIP(hipMemcpy(*d, h, n * sizeof(T), hipMemcpyHostToDevice));
  return GM_OK;
}


// Largest number of nonzeros of one child's nodal interpolation W that the
// Galerkin kernel keeps in LDS (a Q2 child of a Q2 parent: 125 in 3D, 25 in 2D)
template <int DIM>
constexpr int gal_ws_max() { return DIM == 2 ? 32 : 128; }

// Block rows per workgroup of the Galerkin kernel
template <int DIM, int EN>
constexpr int gal_rows() { return DIM == 2 ? DIM + EN : 1; }

// Galerkin coarse operators.  When every finer element lies inside one
// coarser element (its parent) and P maps the parent's unknowns to the
// element's unknowns, R A P = sum over finer elements of P_e^T K_e P_e, with K_e
// the element matrix before Dirichlet rows and P_e the element-local block of
// P.  The coarse element matrix of element E is then the sum over its 2^dim
// children, and the coarse level assembles it like any element matrix
// (the same element-to-nonzero map, its own Dirichlet rows).  P_e is one
// nodal weight matrix W (the same for every nodal variable) and one P1 matrix Q.
static std::string build_galerkin_maps(const gm_ctx *f, const gm_ctx *c, const int *Prow,
                                       const int *Pcol, const double *Pval, MgLevel &L) {
  const int nve = f->nve, np = f->np, nv = f->nv, nch = 1 << f->dim;
  std::vector<int> node_of(c->N, -1);
  for (int n = 0; n < c->num_nodes; n++)
    for (int k = c->first_unknown[n]; k < c->first_unknown[n + 1]; k++) node_of[k] = n;
  std::vector<int> elem_of_centroid(c->num_nodes, -1);
  for (int e = 0; e < c->num_elems; e++) elem_of_centroid[c->elem_centroid[e]] = e;
  std::vector<int> child((size_t)c->num_elems * nch, -1), nchild(c->num_elems, 0);
  std::vector<double> W((size_t)f->num_elems * nve * nve, 0.0);
  std::vector<double> Q((size_t)f->num_elems * np * np, 0.0);
  for (int e = 0; e < f->num_elems; e++) {
    // parent: the coarse element whose centroid node enters the interpolation
    // of this element's centroid
    const int ur = f->first_unknown[f->elem_centroid[e]];
    int parent = -1;
    for (int k = Prow[ur]; k < Prow[ur + 1]; k++) {
      const int pe = elem_of_centroid[node_of[Pcol[k]]];
      if (pe < 0 || Pval[k] == 0.0) continue;
      if (parent >= 0 && parent != pe) return "an element's centroid interpolates from two coarse elements";
      parent = pe;
    }
    if (parent < 0) return "an element has no parent coarse element";
    if (nchild[parent] >= nch) return "a coarse element has more than 2^dim children";
    child[(size_t)parent * nch + nchild[parent]++] = e;
    const int *cn = &c->conn[(size_t)parent * nve];
    for (int i = 0; i < nve; i++) {
      const int u = f->first_unknown[f->conn[(size_t)e * nve + i]];  // first nodal variable
      for (int k = Prow[u]; k < Prow[u + 1]; k++) {
        const int n = node_of[Pcol[k]];
        if (Pcol[k] != c->first_unknown[n]) return "P couples different variables";
        int m = 0;
        while (m < nve && cn[m] != n) m++;
        if (m == nve) return "P couples an element to unknowns outside its parent";
        W[(size_t)e * nve * nve + i * nve + m] = Pval[k];
      }
    }
    const int pf = f->first_unknown[f->elem_centroid[e]] + nv;
    const int pc = c->first_unknown[c->elem_centroid[parent]] + nv;
    for (int kk = 0; kk < np; kk++)
      for (int k = Prow[pf + kk]; k < Prow[pf + kk + 1]; k++) {
        const int l = Pcol[k] - pc;
        if (l < 0 || l >= np) return "P couples pressure outside the parent element";
        Q[(size_t)e * np * np + kk * np + l] = Pval[k];
      }
  }
  for (int e = 0; e < c->num_elems; e++)
    if (nchild[e] != nch) return "a coarse element without 2^dim children";
  // W by columns, nonzeros only (a Q2 child of a Q2 parent: 125 of 729 in 3D)
  int stride = 1;
  for (int e = 0; e < f->num_elems; e++) {
    int nz = 0;
    for (int t = 0; t < nve * nve; t++) nz += W[(size_t)e * nve * nve + t] != 0.0;
    stride = std::max(stride, nz);
  }
  if (stride > (f->dim == 2 ? gal_ws_max<2>() : gal_ws_max<3>()))
    return "a child's nodal interpolation has more nonzeros than the Galerkin kernel keeps";
  std::vector<int> Wp((size_t)f->num_elems * (nve + 1)), Wi((size_t)f->num_elems * stride, 0);
  std::vector<double> Wv((size_t)f->num_elems * stride, 0.0);
  for (int e = 0; e < f->num_elems; e++) {
    const double *We = &W[(size_t)e * nve * nve];
    int k = 0;
    for (int m = 0; m < nve; m++) {
      Wp[(size_t)e * (nve + 1) + m] = k;
      for (int i = 0; i < nve; i++)
        if (We[i * nve + m] != 0.0) {
          Wi[(size_t)e * stride + k] = i;
          Wv[(size_t)e * stride + k] = We[i * nve + m];
          k++;
        }
    }
    Wp[(size_t)e * (nve + 1) + nve] = k;
  }
  L.W_stride = stride;
  if (upv(&L.d_child, child.data(), child.size()) || upv(&L.d_Wp, Wp.data(), Wp.size()) ||
      upv(&L.d_Wi, Wi.data(), Wi.size()) || upv(&L.d_Wv, Wv.data(), Wv.size()) ||
      upv(&L.d_Q, Q.data(), Q.size()))
    return "device allocation failed";
  return "";
}

// One weight of a child's nodal interpolation and the finer node it is for
template <typename CT>
struct alignas(2 * sizeof(CT)) GalW {
  CT w;
  int i;
};

// the n entries of a node pair's row, in 16-byte reads where n allows
template <int n, typename CT>
__device__ inline void load_cols(const CT *p, CT *v) {
  constexpr int W = n * sizeof(CT) % 16 == 0 ? 16 / sizeof(CT) : 1;
  if constexpr (W > 1) {
    typedef CT Wide __attribute__((ext_vector_type(W)));
#pragma unroll
    for (int b = 0; b < n; b += W) {
      const Wide w = *(const Wide *)(p + b);
#pragma unroll
      for (int l = 0; l < W; l++) v[b + l] = w[l];
    }
  } else {
#pragma unroll
    for (int b = 0; b < n; b++) v[b] = p[b];
  }
}

// Coarse element matrices P_e^T K_e P_e summed over the children of each coarse
// element, in the element matrices' layout: nodal block rows a as [i][j][b],
// then momentum x P, continuity x velocity, P x P.
//
// A workgroup takes RW block rows of one coarse element (HEX27: one, QUAD9:
// all), another its pressure couplings: the blocks are independent, and with
// one workgroup for all of them the levels of up to a few hundred elements
// leave most of the chip idle behind 128 rounds of three barriers (64 coarse
// elements with energy, FP64: 57 us against 580).  Per child: K_e's rows from
// memory a child ahead, T = K W over them in LDS, W^T T summed in registers.
// Larger levels are bound by reading the finer element matrices once (1728
// coarse elements with energy, FP32 products: 353 us for 1.4 GB).
template <int DIM, int EN, typename CT>
__global__ __launch_bounds__(256) void k_galerkin(const double *__restrict__ kf,
                                                  const int *__restrict__ child,
                                                  const int *__restrict__ Wp,
                                                  const int *__restrict__ Wi,
                                                  const double *__restrict__ Wv, int ws,
                                                  const double *__restrict__ Q, long long E,
                                                  long long off_mp, double *__restrict__ kc) {
  constexpr int NVE = DIM == 2 ? 9 : 27, NP = DIM + 1, NV = DIM + EN, NCH = 1 << DIM, NT = 256;
  constexpr int NVE2 = NVE * NVE, RW = gal_rows<DIM, EN>(), PARTS = NV / RW + 1;
  constexpr int ROW = NVE * NV, LROW = ROW + (DIM == 3 && sizeof(CT) == 8 ? 2 : 0);  // padded against bank conflicts
  constexpr int NK = RW * NVE2 * NV, RK = (NK + NT - 1) / NT;    // entries of the block rows
  constexpr int NI = RW * NVE2, RN = (NI + NT - 1) / NT;         // node pairs of the block rows
  constexpr int NMP = DIM * NVE * NP;          // momentum x P (= continuity x velocity) entries
  constexpr int NPC = 2 * NMP + NP * NP;       // pressure couplings, contiguous from off_mp
  constexpr int RP = (NPC + NT - 1) / NT;
  constexpr int WSM = gal_ws_max<DIM>();
  // W of every child by columns, loaded once: s_wp[c][m] .. s_wp[c][m + 1]
  // index the finer nodes (ascending) interpolating from coarse node m and
  // their weights, s_w; only these terms of the dense sums are nonzero
  __shared__ alignas(16) CT sK[RW * NVE * LROW];
  __shared__ GalW<CT> s_w[NCH * WSM];
  __shared__ CT sQ[NP * NP];
  __shared__ int s_wp[NCH][NVE + 1];
  static_assert(NPC <= RW * NVE * LROW, "the pressure couplings fit the block rows' space");
  const int ec = blockIdx.x / PARTS, part = blockIdx.x - ec * PARTS, tid = threadIdx.x;
  const int *ch = child + (size_t)ec * NCH;
  double *__restrict__ out = kc + (size_t)ec * E;
  const bool press = part == PARTS - 1;
  const size_t off = press ? (size_t)off_mp : (size_t)part * NK;
  const int cnt = press ? NPC : NK;
  double kr[RK];
  static_assert(RP <= RK, "registers for the pressure couplings");
  auto fetch = [&](int c) {
    const double *Kf = kf + (size_t)ch[c] * E + off;
#pragma unroll
    for (int r = 0; r < RK; r++) {
      const int t = tid + r * NT;
      kr[r] = t < cnt ? Kf[t] : 0.0;
    }
  };
  fetch(0);
  for (int t = tid; t < NCH * (NVE + 1); t += NT) {
    const int c = t / (NVE + 1), m = t - c * (NVE + 1);
    s_wp[c][m] = Wp[(size_t)ch[c] * (NVE + 1) + m];
  }
  for (int t = tid; t < NCH * WSM; t += NT) {
    const int c = t / WSM, k = t - c * WSM;
    if (k < ws) {
      s_w[t].i = Wi[(size_t)ch[c] * ws + k];
      s_w[t].w = (CT)Wv[(size_t)ch[c] * ws + k];
    }
  }
  if (!press) {
    CT acc[RN][NV];
#pragma unroll
    for (int r = 0; r < RN; r++)
#pragma unroll
      for (int b = 0; b < NV; b++) acc[r][b] = 0;
#pragma unroll 1
    for (int c = 0; c < NCH; c++) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < RK; r++) {
        const int t = tid + r * NT, i = t / ROW;
        if (t < NK) sK[i * LROW + t - i * ROW] = (CT)kr[r];
      }
      if (c + 1 < NCH) fetch(c + 1);
      const int *wp = s_wp[c];
      const GalW<CT> *w = s_w + c * WSM;
      __syncthreads();
      CT T[RN][NV];  // T = K W: row i, column m of W
#pragma unroll
      for (int r = 0; r < RN; r++) {
        const int t = tid + r * NT, a = t / NVE2, t2 = t - a * NVE2, m = t2 / NVE, i = t2 - m * NVE;
#pragma unroll
        for (int b = 0; b < NV; b++) T[r][b] = 0;
        if (t < NI)
          for (int k = wp[m]; k < wp[m + 1]; k++) {
            const GalW<CT> x = w[k];
            CT y[NV];
            load_cols<NV>(sK + (a * NVE + i) * LROW + x.i * NV, y);
#pragma unroll
            for (int b = 0; b < NV; b++) T[r][b] += y[b] * x.w;
          }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < RN; r++) {
        const int t = tid + r * NT, a = t / NVE2, t2 = t - a * NVE2, m = t2 / NVE, i = t2 - m * NVE;
        if (t < NI)
#pragma unroll
          for (int b = 0; b < NV; b++) sK[(a * NVE + i) * LROW + m * NV + b] = T[r][b];
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < RN; r++) {  // acc += W^T T: row m, column n
        const int t = tid + r * NT, a = t / NVE2, t2 = t - a * NVE2, m = t2 / NVE, n = t2 - m * NVE;
        if (t >= NI) continue;
        CT v[NV];
#pragma unroll
        for (int b = 0; b < NV; b++) v[b] = 0;
        for (int k = wp[m]; k < wp[m + 1]; k++) {
          const GalW<CT> x = w[k];
          CT y[NV];
          load_cols<NV>(sK + (a * NVE + x.i) * LROW + n * NV, y);
#pragma unroll
          for (int b = 0; b < NV; b++) v[b] += x.w * y[b];
        }
#pragma unroll
        for (int b = 0; b < NV; b++) acc[r][b] += v[b];
      }
    }
#pragma unroll
    for (int r = 0; r < RN; r++) {
      const int t = tid + r * NT;
      if (t < NI)
#pragma unroll
        for (int b = 0; b < NV; b++) out[off + (size_t)t * NV + b] = acc[r][b];
    }
    return;
  }
  CT accp[RP];
#pragma unroll
  for (int r = 0; r < RP; r++) accp[r] = 0.0;
#pragma unroll 1
  for (int c = 0; c < NCH; c++) {
    __syncthreads();
    if (tid < NP * NP) sQ[tid] = (CT)Q[(size_t)ch[c] * NP * NP + tid];
#pragma unroll
    for (int r = 0; r < RP; r++) {
      const int t = tid + r * NT;
      if (t < NPC) sK[t] = (CT)kr[r];
    }
    if (c + 1 < NCH) fetch(c + 1);
    const int *wp = s_wp[c];
    const GalW<CT> *w = s_w + c * WSM;
    __syncthreads();
    // over the nodes first (W^T K, K W; nothing for P x P), then over the P1 dofs
    CT T[RP];
#pragma unroll
    for (int r = 0; r < RP; r++) {
      const int t = tid + r * NT;
      T[r] = 0;
      if (t >= 2 * NMP) continue;
      const bool mp = t < NMP;
      const int node = mp ? t / NP % NVE : (t - NMP) % NVE;
      const int base = mp ? t - node * NP : t - node, step = mp ? NP : 1;
      for (int k = wp[node]; k < wp[node + 1]; k++) T[r] += w[k].w * sK[base + w[k].i * step];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RP; r++) {
      const int t = tid + r * NT;
      if (t < 2 * NMP) sK[t] = T[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RP; r++) {
      const int t = tid + r * NT;
      if (t >= NPC) continue;
      CT v = 0;
      if (t < NMP) {  // row (a, m) momentum, column l pressure
        const int l = t % NP;
#pragma unroll
        for (int k = 0; k < NP; k++) v += sK[t - l + k] * sQ[k * NP + l];
      } else if (t < 2 * NMP) {  // row l continuity, column (b, n) velocity
        const int t2 = t - NMP, l = t2 / NVE % NP;
#pragma unroll
        for (int k = 0; k < NP; k++) v += sQ[k * NP + l] * sK[t + (k - l) * NVE];
      } else {  // P x P
        const int t3 = t - 2 * NMP, l = t3 / NP, l2 = t3 - l * NP;
#pragma unroll
        for (int k = 0; k < NP; k++)
#pragma unroll
          for (int k2 = 0; k2 < NP; k2++)
            v += sQ[k * NP + l] * sK[2 * NMP + k * NP + k2] * sQ[k2 * NP + l2];
      }
      accp[r] += v;
    }
  }
#pragma unroll
  for (int r = 0; r < RP; r++) {
    const int t = tid + r * NT;
    if (t < NPC) out[off_mp + t] = accp[r];
  }
}

template <typename JT>
static int galerkin_level(gm_ctx *prof, const gm_ctx *above, MgLevel &L, JT *val) {
  gm_ctx *lc = L.ctx;
  const ElemLayout &ly = lc->lay;
  const int nch = 1 << lc->dim;
  const double gbytes = ((double)above->num_elems * (ly.total + lc->np * lc->np) +
                         (double)lc->num_elems * ly.total) * 8.0 + 4.0 * nch * lc->num_elems +
                        (double)above->num_elems * (L.W_stride * 12.0 + (lc->nve + 1) * 4.0);
  // products in the precision of the coarse matrices (FP32 under mixed precision)
  using CT = JT;
  auto kern = lc->dim == 2 ? (lc->energy ? k_galerkin<2, 1, CT> : k_galerkin<2, 0, CT>)
                           : (lc->energy ? k_galerkin<3, 1, CT> : k_galerkin<3, 0, CT>);
  const int parts = (lc->dim == 2 ? 1 : lc->nv) + 1;  // workgroups per coarse element
  gm_launch(prof, GM_K_GALERKIN, gbytes, kern, dim3(lc->num_elems * parts), dim3(256), 0, lc->stream,
            above->d_kel, L.d_child, L.d_Wp, L.d_Wi, L.d_Wv, L.W_stride, L.d_Q, ly.total, ly.off_mp,
            lc->d_kel);
  // with the coarse level's own Dirichlet rows
  double *v64 = nullptr;
  float *v32 = nullptr;
  if constexpr (sizeof(JT) == 8) v64 = val;
  else v32 = val;
  return gm_gather(prof, GM_K_ELEM_SCATTER, lc, lc->stream, lc->d_kel, nullptr, v64, v32, 1, nullptr, nullptr,
                   nullptr);
}

int gm_mg_kel_alloc(gm_ctx *c) {
  if (!c->d_kel) GM_HIP(hipMalloc(&c->d_kel, (size_t)c->num_elems * c->lay.total * sizeof(double)));
  return GM_OK;
}

extern "C" int gm_mg_copy_level_matrix(const gm_ctx *c, int level, double *val) {
  if (!c || !val || level < 1 || level > (int)c->mg.size()) return GM_ERR_ARG;
  const MgLevel &L = c->mg[level - 1];
  if (!L.d_val) {
    gm_set_error("multigrid level %d has no matrix yet", level);
    return GM_ERR_ARG;
  }
  const size_t n = L.ctx->nval;
  if (L.d_val == L.d_val_p[1]) {
    std::vector<float> h(n);
    GM_HIP(hipMemcpy(h.data(), L.d_val, n * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < n; i++) val[i] = h[i];
  } else {
    GM_HIP(hipMemcpy(val, L.d_val, n * sizeof(double), hipMemcpyDeviceToHost));
  }
  return GM_OK;
}

extern "C" int gm_mg_copy_block_inverse(const gm_ctx *c, int level, int elem, double *out) {
  if (!c || !out || level < 0 || level > (int)c->mg.size()) return GM_ERR_ARG;
  const MgLevel &L = level == 0 ? c->mg0 : c->mg[level - 1];
  const gm_ctx *lc = level == 0 ? c : L.ctx;
  if (elem < 0 || elem >= lc->num_elems) return GM_ERR_ARG;
  if (!L.d_ainv) {
    gm_set_error("multigrid level %d has no element-block inverses yet", level);
    return GM_ERR_ARG;
  }
  const size_t n = nloc_of(lc), off = (size_t)elem * n * n;
  if (L.d_ainv == L.d_ainv_p[1]) {
    std::vector<float> h(n * n);
    GM_HIP(hipMemcpy(h.data(), (const float *)L.d_ainv + off, n * n * sizeof(float),
                     hipMemcpyDeviceToHost));
    for (size_t i = 0; i < n * n; i++) out[i] = h[i];
  } else {
    GM_HIP(hipMemcpy(out, (const double *)L.d_ainv + off, n * n * sizeof(double),
                     hipMemcpyDeviceToHost));
  }
  return (int)n;
}

extern "C" int gm_mg_copy_coarse_inverse(const gm_ctx *c, double *out) {
  if (!c || !out || c->mg.empty()) return GM_ERR_ARG;
  const MgLevel &L = c->mg.back();
  if (!L.d_dense || L.dense_n != L.ctx->N) {
    gm_set_error("the coarsest multigrid level has no dense inverse yet (no set-up with an "
                 "exact coarse solve)");
    return GM_ERR_ARG;
  }
  const size_t n = (size_t)L.dense_n;
  GM_HIP(hipMemcpy(out, L.d_dense, n * n * sizeof(double), hipMemcpyDeviceToHost));
  return (int)n;
}

extern "C" int gm_mg_add_level(gm_ctx *fine, gm_ctx *coarse, const int *P_rowptr, const int *P_col,
                               const double *P_val, const int *inject) {
  if (!fine || !coarse || !P_rowptr || !P_col || !P_val || !inject) return GM_ERR_ARG;
  gm_ctx *above = fine->mg.empty() ? fine : fine->mg.back().ctx;
  if (coarse->dim != fine->dim || coarse->energy != fine->energy) {
    gm_set_error("coarse level has a different dimension or variable set");
    return GM_ERR_ARG;
  }
  MgLevel L;
  L.ctx = coarse;
  const int Nf = above->N, Nc = coarse->N;
  const int nnz = P_rowptr[Nf];
  for (int k = 0; k < nnz; k++)
    if (P_col[k] < 0 || P_col[k] >= Nc) {
      gm_set_error("prolongation column %d outside the coarse level", P_col[k]);
      return GM_ERR_ARG;
    }
  for (int n = 0; n < coarse->num_nodes; n++)
    if (inject[n] < 0 || inject[n] >= above->num_nodes) {
      gm_set_error("injection map entry outside the finer level");
      return GM_ERR_ARG;
    }
  int rc;
  if ((rc = gm_e2nz_setup(fine)) || (rc = gm_e2nz_setup(coarse))) return rc;
  // R = P^T
  std::vector<int> rrow(Nc + 1, 0), rcol(nnz);
  std::vector<double> rval(nnz);
  for (int k = 0; k < nnz; k++) rrow[P_col[k] + 1]++;
  for (int i = 0; i < Nc; i++) rrow[i + 1] += rrow[i];
  std::vector<int> fp(rrow.begin(), rrow.end() - 1);
  for (int i = 0; i < Nf; i++)
    for (int k = P_rowptr[i]; k < P_rowptr[i + 1]; k++) {
      const int q = fp[P_col[k]]++;
      rcol[q] = i;
      rval[q] = P_val[k];
    }
  if ((rc = upv(&L.d_Prow, P_rowptr, Nf + 1)) || (rc = upv(&L.d_Pcol, P_col, nnz)) ||
      (rc = upv(&L.d_Pval, P_val, nnz)) || (rc = upv(&L.d_Rrow, rrow.data(), Nc + 1)) ||
      (rc = upv(&L.d_Rcol, rcol.data(), nnz)) || (rc = upv(&L.d_Rval, rval.data(), nnz)) ||
      (rc = upv(&L.d_inject, inject, coarse->num_nodes)))
    return rc;
  L.nnz = nnz;
  L.gal_err = build_galerkin_maps(above, coarse, P_rowptr, P_col, P_val, L);
  L.gal_ok = L.gal_err.empty();
  GM_HIP(hipMalloc(&L.d_state, Nc * sizeof(double)));
  GM_HIP(hipMalloc(&L.d_rdummy, Nc * sizeof(double)));
  fine->mg.push_back(L);
  return GM_OK;
}

extern "C" int gm_mg_num_levels(const gm_ctx *c) { return c ? (int)c->mg.size() + 1 : GM_ERR_ARG; }

// Level vectors are FP64 in both precisions; matrices and element-block
// inverses are FP32 in the mixed precision.
static int alloc_level_vectors(MgLevel &L, const gm_ctx *lc, int prec, bool coarse) {
  const size_t N = lc->N;
  const size_t es = prec == GM_PREC_MIXED ? sizeof(float) : sizeof(double);
  if (!L.d_x) {
    GM_HIP(hipMalloc(&L.d_x, N * sizeof(double)));
    GM_HIP(hipMalloc(&L.d_b, N * sizeof(double)));
    GM_HIP(hipMalloc(&L.d_r, N * sizeof(double)));
    L.vec_prec = 0;
  }
  const size_t nl = nloc_of(lc);
  const int pi = prec == GM_PREC_MIXED ? 1 : 0;
  if (!L.d_ainv_p[pi]) GM_HIP(hipMalloc(&L.d_ainv_p[pi], (size_t)lc->num_elems * nl * nl * es));
  L.d_ainv = L.d_ainv_p[pi];
  if (coarse) {
    if (!L.d_val_p[pi]) GM_HIP(hipMalloc(&L.d_val_p[pi], (size_t)lc->nval * es));
    L.d_val = L.d_val_p[pi];
  }
  return GM_OK;
}

template <int DIM, int EN, typename VT, typename AT>
static void launch_invert(gm_ctx *prof, gm_ctx *lc, hipStream_t s, const VT *val, AT *ainv) {
  constexpr int n = Loc<DIM, EN>::N;
  // gathered entries + map + inverses written
  const double bytes = (double)lc->num_elems * n * n * (sizeof(VT) + 4 + sizeof(AT));
  if constexpr (DIM == 3) {
    // 3D blocks (n = 85 / 112) in registers, 16 x 16 threads: three
    // workgroups per CU (164 VGPRs) overlap their pivot steps' barriers
    gm_launch(prof, GM_K_VANKA_INV, bytes, k_vanka_invert_reg<DIM, EN, VT, AT, AT, 16, 16>,
              dim3(lc->num_elems), dim3(256), 0, s, level_dev(lc), val, ainv);
  } else {
    gm_launch(prof, GM_K_VANKA_INV, bytes, k_vanka_invert<DIM, EN, VT, AT, AT>, dim3((lc->num_elems + 7) / 8),
              dim3(256), 0, s, level_dev(lc), lc->num_elems, val, ainv);
  }
}

template <typename VT>
static void invert(gm_ctx *prof, gm_ctx *lc, hipStream_t s, const VT *val, VT *ainv) {
  if (lc->dim == 2) {
    if (lc->energy) launch_invert<2, 1, VT, VT>(prof, lc, s, val, ainv);
    else launch_invert<2, 0, VT, VT>(prof, lc, s, val, ainv);
  } else {
    if (lc->energy) launch_invert<3, 1, VT, VT>(prof, lc, s, val, ainv);
    else launch_invert<3, 0, VT, VT>(prof, lc, s, val, ainv);
  }
}

// Rows touched by each element colour: the unknowns of its elements.
static int build_colour_rows(gm_ctx *lc) {
  if (lc->d_mg_rows) return GM_OK;
  const int nve = lc->nve, cl = lc->dim == 2 ? 8 : 20;
  std::vector<int> rows;
  std::vector<char> seen(lc->N, 0);
  lc->mg_rows_ptr.assign(1, 0);
  lc->mg_rows_nnz.clear();
  for (int col = 0; col < lc->n_ecol; col++) {
    std::vector<int> list;
    for (int k = lc->ecol_ptr[col]; k < lc->ecol_ptr[col + 1]; k++) {
      const int e = lc->ecol_elems[k];
      for (int i = 0; i < nve; i++) {
        const int n = lc->conn[(size_t)e * nve + i];
        const int cnt = (i == cl) ? lc->first_unknown[n + 1] - lc->first_unknown[n] : lc->nv;
        for (int a = 0; a < cnt; a++) list.push_back(lc->first_unknown[n] + a);
      }
    }
    std::sort(list.begin(), list.end());
    list.erase(std::unique(list.begin(), list.end()), list.end());
    long long nnz = 0;
    for (int r : list) nnz += 1 + lc->bindx[r + 1] - lc->bindx[r];
    rows.insert(rows.end(), list.begin(), list.end());
    lc->mg_rows_ptr.push_back((int)rows.size());
    lc->mg_rows_nnz.push_back(nnz);
  }
  // multiplicity of every unknown among the element blocks
  std::vector<double> w(lc->N, 0.0);
  for (int e = 0; e < lc->num_elems; e++)
    for (int i = 0; i < nve; i++) {
      const int n = lc->conn[(size_t)e * nve + i];
      const int cnt = (i == cl) ? lc->first_unknown[n + 1] - lc->first_unknown[n] : lc->nv;
      for (int a = 0; a < cnt; a++) w[lc->first_unknown[n] + a] += 1.0;
    }
  for (double &v : w) v = v > 0.0 ? 1.0 / v : 0.0;
  int rc = upv(&lc->d_mg_wmul, w.data(), w.size());
  if (rc) return rc;
  // gather lists of the additive smoother
  if ((rc = gm_unknown_places(lc))) return rc;
  GM_HIP(hipMalloc(&lc->d_mg_corr, (size_t)lc->num_elems * nloc_of(lc) * sizeof(double)));
  return upv(&lc->d_mg_rows, rows.data(), rows.size());
}

// Dense inverse of the coarsest level's Jacobian (exact coarse solve),
// enqueued on stream s; coarse_inverse_finish waits for it and reports a
// singular matrix.
static int coarse_inverse(gm_ctx *c, MgLevel &L, int prec, hipStream_t s) {
  gm_ctx *lc = L.ctx;
  const int n = lc->N;
  if (n > GM_MG_DIRECT_MAX) {
    gm_set_error("coarsest multigrid level has %d unknowns (exact solve up to %d): coarsen "
                 "further or set mg_coarse_sweeps > 0", n, GM_MG_DIRECT_MAX);
    return GM_ERR_ARG;
  }
  if (L.dense_n != n) {
    for (void *p : {(void *)L.d_dense, (void *)L.d_dense2, (void *)L.d_pcol, (void *)L.d_perm})
      if (p) (void)hipFree(p);
    L.d_dense = L.d_dense2 = L.d_pcol = nullptr;
    L.d_perm = nullptr;
    L.dense_n = 0;
    const size_t cells = (size_t)n * n + GJ_NB;  // a margin: whole panels are read
    GM_HIP(hipMalloc(&L.d_dense, cells * sizeof(double)));
    GM_HIP(hipMalloc(&L.d_dense2, cells * sizeof(double)));
    GM_HIP(hipMalloc(&L.d_pcol, (size_t)2 * GJ_NB * n * sizeof(double)));
    GM_HIP(hipMalloc(&L.d_perm, (size_t)2 * n * sizeof(int)));
    L.dense_n = n;
  }
  // panel width, rows per thread and threads: the panel in registers, up to 64 a thread
  const int pw = n <= 1536 ? 16 : 8, np = (n + pw - 1) / pw;
  const int nt = n <= 768 ? 256 : n <= 1536 ? 512 : 1024;
  auto step = n <= 256    ? k_gjb_step<16, 1, 256>
              : n <= 768  ? k_gjb_step<16, 3, 256>
              : n <= 1536 ? k_gjb_step<16, 3, 512>
                          : k_gjb_step<8, 4, 1024>;
  static_assert(GM_MG_DIRECT_MAX <= 4096 && GJ_NB >= 16, "k_gjb_step's rows and columns");
  // the last of the np launches that write the array writes d_dense2
  double *from = np & 1 ? L.d_dense : L.d_dense2, *to = np & 1 ? L.d_dense2 : L.d_dense;
  const long long nn = (long long)n * n;
  k_set<double><<<1024, 256, 0, s>>>(from, nn, 0.0);
  if (prec == GM_PREC_MIXED)
    k_msr_to_dense<float><<<n, 64, 0, s>>>(n, (const float *)L.d_val, lc->d_bindx, from);
  else
    k_msr_to_dense<double><<<n, 64, 0, s>>>(n, (const double *)L.d_val, lc->d_bindx, from);
  GM_HIP(hipMemsetAsync(c->d_flag + 3, 0, sizeof(int), s));
  const int tiles = ((n + 15) / 16) * ((n + 63) / 64);
  const int blocks = (tiles + nt / 64 - 1) / (nt / 64);
  int *piv = L.d_perm, *stepof = L.d_perm + n;
  for (int k = -1; k < np; k++) {
    // panel k applied to the array, panel k + 1 factored
    const int kb = std::max(k, 0) * pw, nb = k < 0 ? 0 : std::min(pw, n - kb);
    const int kb2 = (k + 1) * pw, nb2 = k + 1 < np ? std::min(pw, n - kb2) : 0;
    double *p0 = L.d_pcol + (size_t)(k & 1) * GJ_NB * n, *p1 = L.d_pcol + (size_t)((k + 1) & 1) * GJ_NB * n;
    // the array read and written, the next panel's columns
    const double bytes = (k < 0 ? 0.0 : 16.0 * (double)nn) + 8.0 * n * nb2;
    gm_launch(c, GM_K_COARSE_INV, bytes, step, dim3(1 + (k < 0 ? 0 : blocks)), dim3(nt), 0, s, n, kb, nb,
              std::min(kb2, n), nb2, (const double *)from, to, (const double *)p0, p1, (const int *)(piv + kb),
              piv + std::min(kb2, n), stepof, c->d_flag);
    if (k >= 0) std::swap(from, to);
  }
  k_gj_permute<<<n, 256, 0, s>>>(n, piv, stepof, L.d_dense2, L.d_dense);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

static int coarse_inverse_finish(gm_ctx *c, hipStream_t s) {
  int flag = 0;
  GM_HIP(hipMemcpyAsync(&flag, c->d_flag + 3, sizeof(int), hipMemcpyDeviceToHost, s));
  GM_HIP(hipStreamSynchronize(s));
  if (flag) {
    gm_set_error("singular Jacobian on the coarsest multigrid level");
    return GM_ERR_PIVOT;
  }
  return GM_OK;
}

// Stream of the overlapped element-block inversions, kept off 1/8 of the CUs.
// The inversions fill every CU they may use (three workgroups of 147-VGPR
// waves each), so a workgroup of another stream is placed only where they
// leave room; the coarsest dense inverse is a chain of small launches, each
// of which waited on a full GPU for the inversions to drain.  The spared CUs
// keep that chain moving beside them.  Without the mask the main stream is
// used.
#ifndef GM_INV_SPARE_DIV
#define GM_INV_SPARE_DIV 8  // CUs spared: 1 in this many (1/16 and 1/12 measured slower)
#endif
static int inv_stream(gm_ctx *c, hipStream_t *out) {
  if (!c->s_inv) {
    int dev = 0, ncu = 0;
    GM_HIP(hipGetDevice(&dev));
    GM_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    hipStream_t s = nullptr;
    if (ncu >= 64) {
      std::vector<uint32_t> mask((size_t)(ncu + 31) / 32, 0u);
      const int keep = ncu - ncu / GM_INV_SPARE_DIV;
      for (int i = 0; i < keep; i++) mask[i / 32] |= 1u << (i % 32);
      if (hipExtStreamCreateWithCUMask(&s, (uint32_t)mask.size(), mask.data()) != hipSuccess) {
        (void)hipGetLastError();
        s = nullptr;
      }
    }
    if (s && (hipEventCreateWithFlags(&c->ev_inv[0], hipEventDisableTiming) != hipSuccess ||
              hipEventCreateWithFlags(&c->ev_inv[1], hipEventDisableTiming) != hipSuccess)) {
      (void)hipGetLastError();
      (void)hipStreamDestroy(s);
      s = nullptr;
    }
    c->s_inv = s ? s : c->stream;
  }
  *out = c->s_inv;
  return GM_OK;
}

// Per Newton step: coarse Jacobians at the injected state, local inverses on
// every level, and the dense inverse of the coarsest level when it is solved
// exactly (coarse_direct).  val / val32 is the level-0 (scaled) matrix, x the
// state.
int gm_mg_setup(gm_ctx *c, const double *x, const double *val, const float *val32, int prec,
                const double *scale, int coarse_direct, int galerkin) {
  c->mg_scale = scale;
  if (c->mg.empty()) {
    gm_set_error("multigrid preconditioner requested but no coarse level attached");
    return GM_ERR_ARG;
  }
  int rc;
  if ((rc = alloc_level_vectors(c->mg0, c, prec, false))) return rc;
  if ((rc = build_colour_rows(c))) return rc;
  for (MgLevel &L : c->mg)
    if ((rc = build_colour_rows(L.ctx))) return rc;
  const double *xs = x;
  gm_ctx *above = c;
  if (galerkin && !c->d_kel) {
    gm_set_error("Galerkin coarse operators need the element matrices of the last assembly");
    return GM_ERR_ARG;
  }
  // The level-0 block inverses need only the level-0 matrix: enqueued first,
  // they run beside the coarse levels' Galerkin products and scatters, which
  // use each coarse level's own stream and synchronise only that stream, and
  // beside the coarsest dense inverse.  Beside a long chain of dense-inverse
  // panels (over 32) they use the stream kept off some CUs, ordered after the
  // main stream's assembly; otherwise the main stream.  With kernel timing on,
  // the set-up runs in order on the main stream instead, so that each
  // launch's measured duration is its own.
  const bool overlap = !c->prof;
  hipStream_t si = c->stream;
  if (overlap && coarse_direct && c->mg.back().ctx->N > 512 && (rc = inv_stream(c, &si)))
    return rc;
  if (si != c->stream) {
    GM_HIP(hipEventRecord(c->ev_inv[0], c->stream));
    GM_HIP(hipStreamWaitEvent(si, c->ev_inv[0], 0));
  }
  // on every return from here, what the main stream queues next (the V-cycles,
  // or the next assembly over the matrix being inverted) waits for the
  // inversions
  struct Join {
    gm_ctx *c;
    hipStream_t si;
    ~Join() {
      if (si == c->stream) return;
      if (hipEventRecord(c->ev_inv[1], si) != hipSuccess ||
          hipStreamWaitEvent(c->stream, c->ev_inv[1], 0) != hipSuccess)
        (void)hipStreamSynchronize(si);
    }
  } join{c, si};
  auto invert0 = [&]() {
    if (prec == GM_PREC_MIXED)
      invert<float>(c, c, si, val32, (float *)c->mg0.d_ainv);
    else
      invert<double>(c, c, si, val, (double *)c->mg0.d_ainv);
  };
  if (overlap) invert0();
  GM_HIP(hipGetLastError());
  for (MgLevel &L : c->mg) {
    if (galerkin) {
      gm_ctx *lc = L.ctx;
      if (!L.gal_ok) {
        gm_set_error("Galerkin coarse operators unavailable: %s", L.gal_err.c_str());
        return GM_ERR_ARG;
      }
      if ((rc = alloc_level_vectors(L, lc, prec, true)) || (rc = gm_mg_kel_alloc(lc))) return rc;
      if ((rc = gm_gather_setup(lc))) return rc;
      rc = prec == GM_PREC_MIXED ? galerkin_level<float>(c, above, L, (float *)L.d_val)
                                 : galerkin_level<double>(c, above, L, (double *)L.d_val);
      if (rc) return rc;
      GM_HIP(hipGetLastError());
      GM_HIP(hipStreamSynchronize(lc->stream));
      above = lc;
      continue;
    }
    gm_ctx *lc = L.ctx;
    if ((rc = alloc_level_vectors(L, lc, prec, true))) return rc;
    k_inject<<<1024, 256, 0, c->stream>>>(lc->num_nodes, L.d_inject, above->d_fu, lc->d_fu, lc->nv,
                                          xs, L.d_state);
    GM_HIP(hipGetLastError());
    GM_HIP(hipStreamSynchronize(c->stream));
    k_set<double><<<256, 256, 0, lc->stream>>>(L.d_rdummy, lc->N, 0.0);
    if (prec == GM_PREC_MIXED) {
      k_set<float><<<2048, 256, 0, lc->stream>>>((float *)L.d_val, lc->nval, 0.0f);
      rc = gm_fill_launch(lc, L.d_state, L.d_rdummy, nullptr, (float *)L.d_val);
    } else {
      k_set<double><<<2048, 256, 0, lc->stream>>>((double *)L.d_val, lc->nval, 0.0);
      rc = gm_fill_launch(lc, L.d_state, L.d_rdummy, (double *)L.d_val, nullptr);
    }
    if (rc) return rc;
    xs = L.d_state;
    above = lc;
  }
  auto invert_coarse = [&]() {
    if (prec == GM_PREC_MIXED) {
      for (MgLevel &L : c->mg)
        invert<float>(c, L.ctx, si, (const float *)L.d_val, (float *)L.d_ainv);
    } else {
      for (MgLevel &L : c->mg)
        invert<double>(c, L.ctx, si, (const double *)L.d_val, (double *)L.d_ainv);
    }
  };
  // The coarse levels' block inverses are queued behind the level-0 ones
  // before the dense inverse's chain of launches: queueing that chain holds the
  // host until most of it has run.  The coarsest level's dense inverse (one
  // workgroup per panel step, latency bound) runs on that level's own stream,
  // beside the element-block inversions; its matrix is complete here (the
  // Galerkin products were synchronised; a rediscretised matrix was filled and
  // checked on the host).
  if (overlap) invert_coarse();
  hipStream_t cs = overlap ? c->mg.back().ctx->stream : c->stream;
  if (coarse_direct && (rc = coarse_inverse(c, c->mg.back(), prec, cs))) return rc;
  if (!overlap) {
    invert0();
    invert_coarse();
  }
  GM_HIP(hipGetLastError());
  // the V-cycles on the main stream read the dense inverse after this host wait
  // and the block inverses after join's event
  if (coarse_direct && (rc = coarse_inverse_finish(c, cs))) return rc;
  return GM_OK;
}

static gm_ctx *g_prof_ctx = nullptr;  // context whose counters the V-cycle feeds

// lanes per row: 2D rows hold ~50-250 entries (8 lanes: 33 vs 36 us per 256^2 residual
// with 16), 3D rows ~500-2100
template <typename VT, typename BT, int G>
static void resid_g(gm_ctx *lc, hipStream_t s, const VT *a, const BT *x, const BT *b, BT *r) {
  const int blocks = (int)(((long long)lc->N * G + 255) / 256);
  const double bytes = (double)(lc->nval - 1) * (sizeof(VT) + 4) + 4.0 * (lc->N + 1) +
                       3.0 * lc->N * sizeof(BT);
  gm_launch(g_prof_ctx, GM_K_MG_RESID, bytes, k_mg_resid<VT, BT, G>, dim3(blocks), dim3(256), 0, s,
            lc->N, a, lc->d_bindx, x, b, r);
}

template <typename VT, typename BT>
static void resid(gm_ctx *lc, hipStream_t s, const VT *a, const BT *x, const BT *b, BT *r) {
  if (lc->dim == 2 || lc->nn_cap > GM_NODE_CAP_MAX) {  // G lanes per row
    if (lc->dim == 3) resid_g<VT, BT, 64>(lc, s, a, x, b, r);
    else resid_g<VT, BT, 8>(lc, s, a, x, b, r);
    return;
  }
  // HEX27: one wave per node (k_msr_nodes)
  using AT = typename std::conditional<sizeof(BT) == 8, double, float>::type;
  const double bytes = (double)(lc->nval - 1) * sizeof(VT) +
                       4.0 * (2.0 * (lc->num_nodes + 1) + lc->N + lc->nn_list.size()) +
                       3.0 * lc->N * sizeof(BT);
  size_t shm;
  const int nw = gm_msr_nodes_shape<AT>(lc->nn_cap, &shm);
  gm_launch(g_prof_ctx, GM_K_MG_RESID, bytes, k_msr_nodes<AT, VT, BT, BT, true>,
            dim3((lc->num_nodes + nw - 1) / nw), dim3(64 * nw), shm, s, lc->num_nodes, lc->dim, lc->nv,
            lc->nn_cap, lc->d_fu, lc->d_nn_ptr, lc->d_nn_cols, lc->d_bindx, a, x, b, r);
}

template <typename VT, typename BT, int G>
static void resid_rows_g(gm_ctx *lc, hipStream_t s, int col, const VT *a, const BT *x, const BT *b,
                         BT *r) {
  const int nr = lc->mg_rows_ptr[col + 1] - lc->mg_rows_ptr[col];
  if (!nr) return;
  const int blocks = (int)(((long long)nr * G + 255) / 256);
  const double nnz_rows = (double)lc->mg_rows_nnz[col];
  const double bytes = nnz_rows * (sizeof(VT) + 4) + nr * (4.0 * 3 + 3.0 * sizeof(BT));
  gm_launch(g_prof_ctx, GM_K_MG_RESID_ROWS, bytes, k_mg_resid_rows<VT, BT, G>, dim3(blocks), dim3(256),
            0, s, nr, (const int *)(lc->d_mg_rows + lc->mg_rows_ptr[col]), a, (const int *)lc->d_bindx,
            x, b, r);
}

template <typename VT, typename BT>
static void resid_rows(gm_ctx *lc, hipStream_t s, int col, const VT *a, const BT *x, const BT *b,
                       BT *r) {
  if (lc->dim == 3) resid_rows_g<VT, BT, 64>(lc, s, col, a, x, b, r);
  else resid_rows_g<VT, BT, 16>(lc, s, col, a, x, b, r);
}

template <int DIM, int EN, typename AT, typename BT>
static void vanka_colour(gm_ctx *lc, hipStream_t s, int col, const AT *ainv, const BT *r, BT *x,
                         double omega, const double *wmul) {
  constexpr int NT = DIM == 2 ? 64 : 128;
  constexpr int n = Loc<DIM, EN>::N;
  const int cnt = lc->ecol_ptr[col + 1] - lc->ecol_ptr[col];
  if (!cnt) return;
  // inverses, element lists/connectivity, residual gathered, x read and written
  const double bytes = (double)cnt * (n * n * sizeof(AT) + 4.0 * (Loc<DIM, EN>::NVE + 2) +
                                      n * 3.0 * sizeof(BT));
  constexpr int EPB = (2 * n <= NT) ? 2 : 1;
  gm_launch(g_prof_ctx, GM_K_VANKA, bytes, k_vanka_update<DIM, EN, AT, BT, NT>, dim3((cnt + EPB - 1) / EPB), dim3(NT),
            0, s, level_dev(lc), cnt, (const int *)(lc->d_ecol_elems + lc->ecol_ptr[col]), ainv, r, x,
            omega, wmul);
}

template <int DIM, int EN, typename AT, typename BT>
static void vanka_additive(gm_ctx *lc, hipStream_t s, const AT *ainv, const BT *r, BT *x, double omega,
                           bool assign) {
  constexpr int NT = DIM == 2 ? 64 : 128;
  constexpr int n = Loc<DIM, EN>::N;
  constexpr int EPB = (2 * n <= NT) ? 2 : 1;
  const int ne = lc->num_elems;
  // inverses, connectivity, residual gathered, corrections written
  const double bytes = (double)ne * (n * n * sizeof(AT) + 4.0 * (Loc<DIM, EN>::NVE + 1) +
                                     n * (sizeof(BT) + 8.0));
  gm_launch(g_prof_ctx, GM_K_VANKA, bytes, k_vanka_corr<DIM, EN, AT, BT, NT>, dim3((ne + EPB - 1) / EPB),
            dim3(NT), 0, s, level_dev(lc), ne, ainv, r, lc->d_mg_corr);
  // lists, corrections, weights, x read and written
  const double gbytes = (double)ne * n * 12.0 + 4.0 * (lc->N + 1) + lc->N * (8.0 + 2.0 * sizeof(BT));
  gm_launch(g_prof_ctx, GM_K_VANKA_GATHER, gbytes, k_vanka_gather<BT>, dim3((lc->N + 255) / 256),
            dim3(256), 0, s, lc->N, (const int *)lc->d_mg_gptr, (const int *)lc->d_mg_gent,
            (const double *)lc->d_mg_corr, (const double *)lc->d_mg_wmul, omega, x, assign ? 1 : 0);
}

// Multiplicative: coloured block Gauss-Seidel, the residual recomputed on each
// colour's rows.  Additive: one residual per sweep, every element's correction
// from it (one launch), then each unknown sums its corrections weighted by
// 1 / elements sharing it (a second launch; no colours needed).  x_zero:
// smoothing from x = 0 (every level's pre-smoothing in the V-cycle): the first
// additive sweep takes b as its residual and assigns its corrections to x,
// whose entries it never reads (the multiplicative smoother gets x cleared).
template <typename VT, typename BT>
static void smooth(gm_ctx *lc, hipStream_t s, const VT *a, const VT *ainv, const BT *b, BT *x, BT *r,
                   int sweeps, double omega, int additive, bool x_zero) {
  for (int it = 0; it < sweeps; it++) {
    if (additive) {
      const BT *rr = r;
      const bool first = it == 0 && x_zero;  // x = 0: residual b, and x is assigned
      if (first) rr = b;
      else resid<VT, BT>(lc, s, a, x, b, r);
      if (lc->dim == 2) {
        if (lc->energy) vanka_additive<2, 1, VT, BT>(lc, s, ainv, rr, x, omega, first);
        else vanka_additive<2, 0, VT, BT>(lc, s, ainv, rr, x, omega, first);
      } else {
        if (lc->energy) vanka_additive<3, 1, VT, BT>(lc, s, ainv, rr, x, omega, first);
        else vanka_additive<3, 0, VT, BT>(lc, s, ainv, rr, x, omega, first);
      }
      continue;
    }
    const double *w = nullptr;
    for (int col = 0; col < lc->n_ecol; col++) {
      resid_rows<VT, BT>(lc, s, col, a, x, b, r);
      if (lc->dim == 2) {
        if (lc->energy) vanka_colour<2, 1, VT, BT>(lc, s, col, ainv, r, x, omega, w);
        else vanka_colour<2, 0, VT, BT>(lc, s, col, ainv, r, x, omega, w);
      } else {
        if (lc->energy) vanka_colour<3, 1, VT, BT>(lc, s, col, ainv, r, x, omega, w);
        else vanka_colour<3, 0, VT, BT>(lc, s, col, ainv, r, x, omega, w);
      }
    }
  }
}

// z = M^-1 v: one V-cycle.  VT: matrix / inverse type, BT: vector type.
template <typename BT>
static void transfer(gm_ctx *c, hipStream_t s, int nrows, const int *rp, const int *ci,
                     const double *cv, int nnz, int ncols, const BT *v, const double *sc,
                     const signed char *mask, BT *y, int acc) {
  const double bytes = (double)nnz * 12.0 + 4.0 * (nrows + 1) + (double)ncols * sizeof(BT) +
                       (double)nrows * (1 + (acc ? 2 : 1) * sizeof(BT));
  const double avg = nrows ? (double)nnz / nrows : 0.0;  // entries per row
  auto launch = [&](auto kern, int G) {
    gm_launch(c, GM_K_TRANSFER, bytes, kern, dim3((int)(((long long)nrows * G + 255) / 256)), dim3(256),
              0, s, nrows, rp, ci, cv, v, sc, mask, y, acc);
  };
  if (avg <= 4.0) launch(k_csr_apply<BT, 4>, 4);
  else if (avg <= 12.0) launch(k_csr_apply<BT, 8>, 8);
  else launch(k_csr_apply<BT, 16>, 16);
}

template <typename VT, typename BT>
static void vcycle(gm_ctx *c, const VT *a0, const BT *v, BT *z, const gm_solver_opts *o) {
  hipStream_t s = c->stream;
  g_prof_ctx = c;
  const int nl = (int)c->mg.size();
  const int nu = o->mg_nu > 0 ? o->mg_nu : 1;
  const double om = o->mg_omega > 0 ? o->mg_omega : 1.0;
  const int cs = o->mg_coarse_sweeps;  // 0: exact solve with the dense inverse
  auto lv_ctx = [&](int l) { return l == 0 ? c : c->mg[l - 1].ctx; };
  auto lv = [&](int l) -> MgLevel & { return l == 0 ? c->mg0 : c->mg[l - 1]; };
  auto amat = [&](int l) -> const VT * { return l == 0 ? a0 : (const VT *)c->mg[l - 1].d_val; };
  // level 0 works on the caller's vectors
  BT *x0 = z;
  const BT *b0 = v;
  for (int l = 0; l <= nl; l++) {
    gm_ctx *lc = lv_ctx(l);
    MgLevel &L = lv(l);
    BT *x = l == 0 ? x0 : (BT *)L.d_x;
    const BT *b = l == 0 ? b0 : (const BT *)L.d_b;
    if (l == nl && cs <= 0 && L.dense_n == lc->N) {
      const int n = lc->N;
      gm_launch(c, GM_K_MG_DENSE, (double)n * n * 8.0 + 2.0 * n * sizeof(BT), k_dense_gemv<BT>,
                dim3((unsigned)(((long long)n * 64 + 255) / 256)), dim3(256), 0, s, n,
                (const double *)L.d_dense, b, x);
      break;
    }
    // pre-smoothing from x = 0 (the additive smoother's first sweep assigns x)
    if (o->mg_smoother != 1) k_set<BT><<<1024, 256, 0, s>>>(x, lc->N, (BT)0);
    smooth<VT, BT>(lc, s, amat(l), (const VT *)L.d_ainv, b, x, (BT *)L.d_r,
                   l == nl ? (cs > 0 ? cs : 20) : nu, om, o->mg_smoother == 1, true);
    if (l == nl) break;
    resid<VT, BT>(lc, s, amat(l), x, b, (BT *)L.d_r);
    MgLevel &C = c->mg[l];
    // restrict the (unscaled) residual: the level-0 matrix is row-sum scaled
    transfer<BT>(c, s, C.ctx->N, C.d_Rrow, C.d_Rcol, C.d_Rval, C.nnz, lc->N, (const BT *)L.d_r,
                 l == 0 ? c->mg_scale : nullptr, C.ctx->d_dbc, (BT *)C.d_b, 0);
  }
  for (int l = nl - 1; l >= 0; l--) {
    gm_ctx *lc = lv_ctx(l);
    MgLevel &L = lv(l);
    MgLevel &C = c->mg[l];
    BT *x = l == 0 ? x0 : (BT *)L.d_x;
    const BT *b = l == 0 ? b0 : (const BT *)L.d_b;
    transfer<BT>(c, s, lc->N, C.d_Prow, C.d_Pcol, C.d_Pval, C.nnz, C.ctx->N, (const BT *)C.d_x,
                 nullptr, lc->d_dbc, x, 1);
    smooth<VT, BT>(lc, s, amat(l), (const VT *)L.d_ainv, b, x, (BT *)L.d_r, nu, om,
                   o->mg_smoother == 1, false);
  }
}

int gm_mg_apply_d(gm_ctx *c, const double *a0, const double *v, double *z, const gm_solver_opts *o) {
  vcycle<double, double>(c, a0, v, z, o);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

int gm_mg_apply_f(gm_ctx *c, const float *a0, const double *v, double *z, const gm_solver_opts *o) {
  vcycle<float, double>(c, a0, v, z, o);
  GM_HIP(hipGetLastError());
  return GM_OK;
}

void gm_mg_free(gm_ctx *c) {
  auto fr = [](MgLevel &L) {
    void *p[] = {L.d_Prow, L.d_Pcol, L.d_Pval, L.d_Rrow, L.d_Rcol, L.d_Rval, L.d_inject,
                 L.d_state, L.d_rdummy, L.d_x, L.d_b, L.d_r, L.d_val_p[0], L.d_val_p[1],
                 L.d_ainv_p[0], L.d_ainv_p[1],
                 L.d_dense, L.d_dense2, L.d_pcol, L.d_perm, L.d_child, L.d_Wp, L.d_Wi, L.d_Wv, L.d_Q};
    for (void *q : p)
      if (q) (void)hipFree(q);
  };
  for (MgLevel &L : c->mg) fr(L);
  fr(c->mg0);
  c->mg.clear();
  c->mg0 = MgLevel();
}

extern "C" int gm_mg_setup_dev(gm_ctx *c, const double *x, const double *val, const double *scale) {
  if (!c || !x || !val) return GM_ERR_ARG;
  int rc = gm_mg_setup(c, x, val, nullptr, GM_PREC_FP64, scale, 1, 0);
  if (rc) return rc;
  GM_HIP(hipStreamSynchronize(c->stream));
  return GM_OK;
}
