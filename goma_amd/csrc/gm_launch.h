// Kernel launch with per-family timing, for the .hip translation units.
//
// Every launch adds its algorithmic bytes to its family's total.  One launch
// in prof_every (and the family's first) is timed: the dispatch packet itself
// carries the start/stop events (hipExtLaunchKernel), so the measured
// duration is the kernel's execution alone, without the queueing latency that
// a pair of hipEventRecord markers around the launch would add.
#pragma once

#include <hip/hip_ext.h>

#include "gm_internal.h"

// Workgroups of a 1D grid are dispatched round-robin to the 8 XCDs, each with
// its own L2.  Element kernels remap blockIdx.x so that every XCD works
// through one contiguous range of an element list: neighbouring elements,
// which share nodes, then share an L2 (measured: a few per cent on the
// element-block smoother, about 1 % on the HEX27 node-row kernel; neutral to
// slower on the per-row kernels, which keep the plain order).  A bijection on
// [0, gridDim.x).
__device__ inline int xcd_block() {
  const int nb = gridDim.x, b = blockIdx.x;
  const int q = nb >> 3, r = nb & 7, x = b & 7;
  return x * q + min(x, r) + (b >> 3);
}

// sum_k a[k] x[col[k]] over k = k0 + lane, k0 + lane + G, ... < k1, with two
// independent accumulators (two loads in flight per lane).
template <typename AT, typename VT, typename XT, int G>
__device__ inline AT row_dot(const VT *__restrict__ a, const int *__restrict__ col,
                             const XT *__restrict__ x, int k0, int k1, int lane) {
  AT s0 = 0, s1 = 0;
  int k = k0 + lane;
  for (; k + G < k1; k += 2 * G) {
    s0 += (AT)a[k] * (AT)x[col[k]];
    s1 += (AT)a[k + G] * (AT)x[col[k + G]];
  }
  if (k < k1) s0 += (AT)a[k] * (AT)x[col[k]];
  return s0 + s1;
}

// v from the lane R places along in the same row of 16 lanes (DPP row_ror)
template <int R>
__device__ inline int row_ror_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x120 + R, 0xf, 0xf, false);
}
template <int R>
__device__ inline float row_ror_f(float v) {
  return __builtin_bit_cast(float, row_ror_i<R>(__builtin_bit_cast(int, v)));
}
template <int R>
__device__ inline double row_ror_f(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)row_ror_i<R>((int)(unsigned)b);
  const unsigned hi = (unsigned)row_ror_i<R>((int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// maximum over the 16 lanes of a DPP row, in every lane
__device__ inline unsigned row_max16(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));  // row_ror:8
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false));
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false));
}

// of 64 bits: of the high words, then of their low words
__device__ inline unsigned long long row_max16(unsigned long long v) {
  const unsigned hi = (unsigned)(v >> 32), m = row_max16(hi);
  return (unsigned long long)m << 32 | row_max16(hi == m ? (unsigned)v : 0u);
}

// the value of lane j of each DPP row of 16, in all of its lanes (row_newbcast)
template <int j>
__device__ inline double row_bcast_c(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  return __builtin_bit_cast(double, (unsigned long long)__builtin_amdgcn_update_dpp(0ull, b, 0x150 + j, 0xf, 0xf, true));
}
template <int j>
__device__ inline float row_bcast_c(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + j, 0xf, 0xf, true));
}
template <typename T>
__device__ __forceinline__ T row_bcast(T v, int j) {
  switch (j) {
#define GM_B(k) case k: return row_bcast_c<k>(v);
    GM_B(0) GM_B(1) GM_B(2) GM_B(3) GM_B(4) GM_B(5) GM_B(6) GM_B(7)
    GM_B(8) GM_B(9) GM_B(10) GM_B(11) GM_B(12) GM_B(13) GM_B(14)
#undef GM_B
    default: return row_bcast_c<15>(v);
  }
}

// 1 / v, rounded, for every v (subnormal and infinite ones too), 0 for 0
__device__ inline double reciprocal(double v) { return v != 0.0 ? 1.0 / v : 0.0; }
__device__ inline float reciprocal(float v) { return v != 0.0f ? 1.0f / v : 0.0f; }

// inclusive prefix sum over the wave (DPP row shifts, then the row totals)
__device__ inline int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true);   // row_bcast:15
  return v + __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true);  // row_bcast:31
}

// The rows of the MSR matrix one node at a time, without reading a column
// index per nonzero.  Row u of node n holds, for every neighbour node m of n
// in ascending order (n itself included), the unknowns of m in ascending
// order, minus the P columns in an energy row (the interaction mask) and
// minus u itself (the diagonal, stored apart): the order
// find_MSR_problem_graph builds (src/mm_fill_util.c:3229-3445).  One wave per
// node copies the vector's entries at the node's columns to LDS from its
// neighbour list (one lane per neighbour, offsets by a wave prefix sum of the
// neighbours' unknown counts), with the energy row's places among them.  It
// then takes the node's rows four at a time, 16 lanes (one DPP row) per row,
// two neighbouring entries per lane and load, and a reduction by DPP row
// rotations; entry e of row r is place e, or e + 1 from the diagonal's place
// on.  The node graph costs 4 bytes per neighbour for all the node's rows
// instead of 4 bytes per nonzero, and a vector entry is gathered once per node.
// Bound by the values' bytes, and for small rows by the chain of loads that ends
// in them: the first values leave before the neighbour list is read, up to
// four loads of 16 bytes (FP32: 8) per lane stay in flight, and the list holds
// the neighbours' first columns, so nothing is looked up per neighbour.  19^3
// with energy, FP64: 114 us (4.3 TB/s of 5.1 a copy reaches) against 140 with
// column places in LDS, one gather per nonzero and two 8-byte loads in flight;
// 24^3, FP32 values: 155 against 197.  Six waves per SIMD: with 86 VGPRs, five,
// 121 us.  16-byte loads of FP32 values are slower (the rows' ragged ends).  Slower at 48^3 in the older form: the node's
// rows in turn with 64 lanes each (one row's loads in flight at a time), 64
// lanes per row with the column list, a workgroup per node with a row per
// wave, the node's rows walked as one block with per-entry row selection.
// `cap` is the longest pattern of the mesh (LDS: cap + 1 entries and places
// per wave).  RESID: y = b - A x; otherwise y = A x.
template <typename AT, typename VT, typename XT, typename YT, bool RESID>
__global__ __launch_bounds__(256, 6) void k_msr_nodes(int num_nodes, int dim, int nvn, int cap,
                                                   const int *__restrict__ fu,
                                                   const int *__restrict__ nn_ptr,
                                                   const int *__restrict__ nn_cols,
                                                   const int *__restrict__ bindx,
                                                   const VT *__restrict__ a,
                                                   const XT *__restrict__ x,
                                                   const XT *__restrict__ b, YT *__restrict__ y) {
  constexpr int U = 4, MAXU = 8;  // loads in flight; unknowns of a node (HEX27: 4 nodal, 4 of P)
  typedef VT Two __attribute__((ext_vector_type(2), aligned(sizeof(VT))));
  typedef XT XTwo __attribute__((ext_vector_type(2), aligned(sizeof(XT))));
  extern __shared__ double s_pat[];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int n = xcd_block() * nw + w;
  const bool valid = n < num_nodes;
  AT *X = (AT *)s_pat + (size_t)w * (cap + 1);
  unsigned short *PT = (unsigned short *)((AT *)s_pat + (size_t)nw * (cap + 1)) + (size_t)w * (cap + 1);
  const int g = lane >> 4, l = lane & 15;
  int f0 = 0, nu = 0, selfA = 0, selfT = 0, endA = 0, endT = 0, k0 = 0, len = 0;
  Two v[U];
  // entries 2 l + 32 i, + 1 of this lane's row, from entry e0 on
  auto fetch = [&](int e0) {
#pragma unroll
    for (int i = 0; i < U; i++) {
      const int e = e0 + 32 * i + 2 * l;
      v[i] = Two{0, 0};
      if (e + 1 < len) v[i] = *(const Two *)(a + k0 + e);
      else if (e < len) v[i][0] = a[k0 + e];
    }
  };
  auto open = [&](int r) {  // the row's place in the matrix, its first loads
    k0 = len = 0;
    if (r < nu) {
      k0 = bindx[f0 + r];
      len = bindx[f0 + r + 1] - k0;
    }
    fetch(0);
  };
  if (valid) {
    f0 = fu[n];
    nu = fu[n + 1] - f0;
    const int j0 = nn_ptr[n], nb = nn_ptr[n + 1] - j0;
    int first = lane < nb ? nn_cols[j0 + lane] : -2;
    open(g);
    int carry = 0;  // places so far: of all columns, and in the high half of the energy row's
    for (int c0 = 0; c0 < nb; c0 += 64) {
      // first column of the neighbour, twice, plus 1 when it has P columns
      if (c0) first = c0 + lane < nb ? nn_cols[j0 + c0 + lane] : -2;
      const int fm = first >> 1, lenT = first >= 0 ? nvn : 0, lm = lenT + (first > 0 ? (first & 1) * (dim + 1) : 0);
      const int own = lm | lenT << 16;
      XT xm[MAXU];
#pragma unroll
      for (int q = 0; q < MAXU; q += 2) {
        xm[q] = xm[q + 1] = (XT)0;
        if (q + 1 < lm) {
          const XTwo t = *(const XTwo *)(x + fm + q);
          xm[q] = t[0];
          xm[q + 1] = t[1];
        } else if (q < lm) {
          xm[q] = x[fm + q];
        }
      }
      const int inc = wave_scan(own), off = carry + inc - own, offA = off & 0xffff, offT = off >> 16;
#pragma unroll
      for (int q = 0; q < MAXU; q++) {
        if (q < lm) X[offA + q] = (AT)xm[q];
        if (q < lenT) PT[offT + q] = (unsigned short)(offA + q);
      }
      const unsigned long long sb = __ballot(fm == f0);
      if (sb) {
        const int so = __shfl(off, __builtin_ctzll(sb));
        selfA = so & 0xffff;
        selfT = so >> 16;
      }
      carry += __shfl(inc, 63);
    }
    // a zero past the end, for the last loads' missing entries
    endA = carry & 0xffff;
    endT = carry >> 16;
    if (lane == 0) {
      X[endA] = 0;
      PT[endT] = (unsigned short)endA;
    }
  }
  if (!valid) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own LDS
  const bool energy = nvn > dim;
  for (int r0 = 0; r0 < nu; r0 += 4) {
    const int r = r0 + g;
    if (r0) open(r);
    const bool tr = energy && r == dim;
    const int hole = (tr ? selfT : selfA) + r, end = tr ? endT : endA;
    AT s0 = 0, s1 = 0;
    // the longest of the four rows, for all of them
    int last = len;
    last = max(last, __shfl_xor(last, 16));
    last = max(last, __shfl_xor(last, 32));
    for (int e0 = 0; e0 < last; e0 += 32 * U) {
      Two c[U];
#pragma unroll
      for (int i = 0; i < U; i++) c[i] = v[i];
      if (e0 + 32 * U < last) fetch(e0 + 32 * U);
      int p[2 * U];  // places: of all of them, then the energy row's own, then the products
#pragma unroll
      for (int i = 0; i < U; i++) {
        const int e = e0 + 32 * i + 2 * l;
        p[2 * i] = min(e + (e >= hole ? 1 : 0), end);
        p[2 * i + 1] = min(e + 1 + (e + 1 >= hole ? 1 : 0), end);
      }
      if (tr) {
#pragma unroll
        for (int i = 0; i < 2 * U; i++) p[i] = PT[p[i]];
      }
#pragma unroll
      for (int i = 0; i < U; i++) {
        s0 += (AT)c[i][0] * X[p[2 * i]];
        s1 += (AT)c[i][1] * X[p[2 * i + 1]];
      }
    }
    AT t = s0 + s1;
    t += row_ror_f<8>(t);
    t += row_ror_f<4>(t);
    t += row_ror_f<2>(t);
    t += row_ror_f<1>(t);
    if (l == 0 && r < nu) {
      const int u = f0 + r;
      const AT d = (AT)a[u] * X[selfA + r];
      y[u] = RESID ? (YT)((AT)b[u] - t - d) : (YT)(t + d);
    }
  }
}

// Waves per workgroup and LDS bytes of k_msr_nodes
template <typename AT>
static inline int gm_msr_nodes_shape(int cap, size_t *shm) {
  const size_t wave = (size_t)(cap + 1) * (sizeof(AT) + 2);
  const int nw = 4 * wave <= 64 * 1024 ? 4 : 2;
  *shm = nw * wave;
  return nw;
}

template <typename... P, typename... A>
static inline void gm_launch(gm_ctx *pc, int id, double bytes, void (*kern)(P...), dim3 grid,
                             dim3 block, size_t shm, hipStream_t s, A... args) {
  static_assert(sizeof...(P) == sizeof...(A), "kernel argument count");
  hipEvent_t eb = nullptr, ee = nullptr;
  if (pc && gm_prof_take(pc, id, bytes, &eb, &ee))
    hipExtLaunchKernelGGL(kern, grid, block, (std::uint32_t)shm, s, eb, ee, 0u, ((P)args)...);
  else
    kern<<<grid, block, shm, s>>>(((P)args)...);
}
