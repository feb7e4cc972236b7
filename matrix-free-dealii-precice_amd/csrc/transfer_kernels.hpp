// Geometric multigrid transfer between nested hex levels (MGTransferMatrixFree
// as used at mf_elasticity.h:863-877, 920-922 and heat_transfer.h:761-762):
// prolongation is the embedding of the coarse FE space (values of the coarse
// function at the fine support points), restriction its exact transpose, and
// interpolation the nodal interpolant of a fine function on the coarse level.
//
// One workgroup per coarse cell.  The (2p+1)^3 fine support points inside a
// coarse cell form a lattice; the 1D embedding matrix E[(2p+1) x (p+1)] is
// applied in three LDS sweeps.  Every fine lattice entry carries the fine node
// index, the fine constraint bits (28..30) and an owner bit (31): exactly one
// coarse cell owns each fine node, so prolongation adds each fine value once
// without atomics, and restriction counts each fine value once.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "cell_kernels.hpp"

namespace mfg {

constexpr uint32_t kOwnerBit = 1u << 31;
constexpr uint32_t kFineNodeMask = (1u << 28) - 1u;

template <typename CN, typename FN>
struct TransferArgs {
  const uint32_t *coarse_nodes;  // coarse map (stored cell order), constraint bits
  const uint32_t *lattice;       // (2p+1)^3 per coarse cell, same cell order
  int cell_begin, cell_end;
  const double *E;               // (2p+1) x (p+1), row-major
  const CN *coarse_in;
  CN *coarse_out;
  const FN *fine_in;
  FN *fine_out;
  // restriction in one launch: every (coarse cell, point) stores its value at
  // slots[cell N^3 + point] (slots null: in point order) of contrib
  double *contrib;
  const uint32_t *slots;
};

// LDS doubles one coarse cell needs (the largest of the three transfers) with
// KC components at a time
template <int P, int KC = 1>
constexpr int transfer_lds() {
  constexpr int N = P + 1, M = 2 * P + 1;
  return M * N + KC * (M * M * M + M * M * N + M * N * N);
}
// LDS doubles of the prolongation alone
template <int P, int KC>
constexpr int prolongate_lds() {
  constexpr int N = P + 1, M = 2 * P + 1;
  return M * N + KC * (N * N * N + M * N * N + M * M * N);
}
// components at a time of the single-operator kernels: all of them where the
// scratch stays within 64 KB (4 barriers per cell instead of 4 per component,
// the lattice read once).  The prolongation needs less: 33 KB for the three
// components of Q5, 52 KB for Q6.  Prolongation to 32x32x24 cells FP32, one
// component at a time, three in the restriction's LDS, three in its own: Q5 58,
// 62 and 42 us, Q6 98, (too large) and 80; FP64 Q5 101 -> 49, Q6 173 -> 87.
template <int P, int NC>
constexpr int transfer_components() {
  return transfer_lds<P, NC>() * 8 <= 65536 ? NC : 1;
}
template <int P, int NC>
constexpr int prolongate_components() {
  return prolongate_lds<P, NC>() * 8 <= 65536 ? NC : 1;
}

// KC components from `c` on of a node
template <int KC, int NC, typename T>
__device__ inline void load_components(const T *v, int64_t node, int c, double (&out)[KC]) {
  if constexpr (KC == NC) {
    const NodeValues<T, NC> x = load_node<T, NC>(v + node * NC);
#pragma unroll
    for (int k = 0; k < NC; ++k) out[k] = (double)x.v[k];
  } else {
    static_assert(KC == 1, "one component or all");
    out[0] = (double)v[node * NC + c];
  }
}

// The per-cell bodies run on all threads of a workgroup (strided loops; the
// sizes are small and vary with p) and use `lds` as scratch.
template <int P, int NC, typename CN, typename FN, int KC = 1>
__device__ inline void prolongate_cell(const TransferArgs<CN, FN> &a, int cell, double *lds) {
  constexpr int N = P + 1, M = 2 * P + 1, N3 = N * N * N, M3 = M * M * M, S1 = M * N * N, S2 = M * M * N;
  double *sE = lds, *su = sE + M * N, *t1 = su + KC * N3, *t2 = t1 + KC * S1;
  const int t = threadIdx.x, nt = blockDim.x;
  for (int x = t; x < M * N; x += nt) sE[x] = a.E[x];
  for (int c = 0; c < NC; c += KC) {
    __syncthreads();
    for (int x = t; x < N3; x += nt) {
      const uint32_t e = a.coarse_nodes[(int64_t)cell * N3 + x];
      double v[KC];
      load_components<KC, NC>(a.coarse_in, (int64_t)(e & kNodeMaskDev), c, v);
#pragma unroll
      for (int k = 0; k < KC; ++k) su[k * N3 + x] = ((e >> (kConstraintShift + c + k)) & 1u) ? 0.0 : v[k];
    }
    __syncthreads();
    for (int y = t; y < KC * S1; y += nt) {  // t1[I][b][c'] (I fastest)
      const int k = y / S1, x = y - k * S1, I = x % M, bc = x / M;
      double s = 0;
      for (int q = 0; q < N; ++q) s += sE[I * N + q] * su[k * N3 + q + N * bc];
      t1[y] = s;
    }
    __syncthreads();
    for (int y = t; y < KC * S2; y += nt) {  // t2[I][J][c']
      const int k = y / S2, x = y - k * S2, I = x % M, J = (x / M) % M, cz = x / (M * M);
      double s = 0;
      for (int q = 0; q < N; ++q) s += sE[J * N + q] * t1[k * S1 + I + M * (q + N * cz)];
      t2[y] = s;
    }
    __syncthreads();
    for (int x = t; x < M3; x += nt) {
      const uint32_t e = a.lattice[(int64_t)cell * M3 + x];
      if (!(e & kOwnerBit)) continue;
      const int IJ = x % (M * M), K = x / (M * M);
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        if ((e >> (kConstraintShift + c + k)) & 1u) continue;
        double s = 0;
        for (int q = 0; q < N; ++q) s += sE[K * N + q] * t2[k * S2 + IJ + M * M * q];
        FN *dst = a.fine_out + (int64_t)(e & kFineNodeMask) * NC + c + k;
        *dst = (FN)((double)*dst + s);
      }
    }
  }
}

// coarse += P^T fine on one coarse cell (callers run one colour at a time), or
// (kToContrib) the cell's part of it stored per point
template <int P, int NC, typename CN, typename FN, int KC = 1, bool kToContrib = false>
__device__ inline void restrict_cell(const TransferArgs<CN, FN> &a, int cell, double *lds) {
  constexpr int N = P + 1, M = 2 * P + 1, N3 = N * N * N, M3 = M * M * M, S1 = M * N * N, S2 = M * M * N;
  double *sE = lds, *sf = sE + M * N, *t2 = sf + KC * M3, *t1 = t2 + KC * S2;
  const int t = threadIdx.x, nt = blockDim.x;
  for (int x = t; x < M * N; x += nt) sE[x] = a.E[x];
  for (int c = 0; c < NC; c += KC) {
    __syncthreads();
    for (int x = t; x < M3; x += nt) {
      const uint32_t e = a.lattice[(int64_t)cell * M3 + x];
      double v[KC] = {};
      if (e & kOwnerBit) load_components<KC, NC>(a.fine_in, (int64_t)(e & kFineNodeMask), c, v);
#pragma unroll
      for (int k = 0; k < KC; ++k) sf[k * M3 + x] = ((e >> (kConstraintShift + c + k)) & 1u) ? 0.0 : v[k];
    }
    __syncthreads();
    for (int y = t; y < KC * S2; y += nt) {  // t2[I][J][k]
      const int cc = y / S2, x = y - cc * S2, IJ = x % (M * M), k = x / (M * M);
      double s = 0;
      for (int q = 0; q < M; ++q) s += sE[q * N + k] * sf[cc * M3 + IJ + M * M * q];
      t2[y] = s;
    }
    __syncthreads();
    for (int y = t; y < KC * S1; y += nt) {  // t1[I][j][k]
      const int cc = y / S1, x = y - cc * S1, I = x % M, j = (x / M) % N, k = x / (M * N);
      double s = 0;
      for (int q = 0; q < M; ++q) s += sE[q * N + j] * t2[cc * S2 + I + M * (q + M * k)];
      t1[y] = s;
    }
    __syncthreads();
    for (int x = t; x < N3; x += nt) {
      const int64_t q0 = (int64_t)cell * N3 + x;
      const int i = x % N, jk = x / N;
      double s[KC];
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        s[k] = 0;
        for (int q = 0; q < M; ++q) s[k] += sE[q * N + i] * t1[k * S1 + q + M * jk];
      }
      if constexpr (kToContrib) {
        double *dst = a.contrib + (int64_t)(a.slots ? a.slots[q0] : (uint32_t)q0) * NC + c;
#pragma unroll
        for (int k = 0; k < KC; ++k) dst[k] = s[k];
      } else {
        const uint32_t e = a.coarse_nodes[q0];
#pragma unroll
        for (int k = 0; k < KC; ++k) {
          if ((e >> (kConstraintShift + c + k)) & 1u) continue;
          CN *dst = a.coarse_out + (int64_t)(e & kNodeMaskDev) * NC + c + k;
          *dst = (CN)((double)*dst + s[k]);
        }
      }
    }
  }
}

// coarse = nodal interpolant of the fine function; E here is the
// interpolation matrix (p+1) x (2p+1).  Shared coarse nodes receive
// bit-identical values from every cell containing them.
template <int P, int NC, typename CN, typename FN>
__device__ inline void interpolate_cell(const TransferArgs<CN, FN> &a, int cell, double *lds) {
  constexpr int N = P + 1, M = 2 * P + 1, N3 = N * N * N, M3 = M * M * M;
  double *sI = lds, *sf = sI + N * M, *t2 = sf + M3, *t1 = t2 + M * M * N;
  const int t = threadIdx.x, nt = blockDim.x;
  for (int x = t; x < N * M; x += nt) sI[x] = a.E[x];
  for (int c = 0; c < NC; ++c) {
    __syncthreads();
    for (int x = t; x < M3; x += nt) {
      const uint32_t e = a.lattice[(int64_t)cell * M3 + x];
      sf[x] = (double)a.fine_in[(int64_t)(e & kFineNodeMask) * NC + c];
    }
    __syncthreads();
    for (int x = t; x < M * M * N; x += nt) {  // t2[I][J][k]
      const int IJ = x % (M * M), k = x / (M * M);
      double s = 0;
      for (int q = 0; q < M; ++q) s += sI[k * M + q] * sf[IJ + M * M * q];
      t2[x] = s;
    }
    __syncthreads();
    for (int x = t; x < M * N * N; x += nt) {
      const int I = x % M, j = (x / M) % N, k = x / (M * N);
      double s = 0;
      for (int q = 0; q < M; ++q) s += sI[j * M + q] * t2[I + M * (q + M * k)];
      t1[x] = s;
    }
    __syncthreads();
    for (int x = t; x < N3; x += nt) {
      const uint32_t e = a.coarse_nodes[(int64_t)cell * N3 + x];
      const int i = x % N, jk = x / N;
      double s = 0;
      for (int q = 0; q < M; ++q) s += sI[i * M + q] * t1[q + M * jk];
      a.coarse_out[(int64_t)(e & kNodeMaskDev) * NC + c] = (CN)s;
    }
  }
}

// One workgroup of 256 threads per coarse cell of [cell_begin, cell_end).
template <int P, int NC, typename CN, typename FN>
__global__ void __launch_bounds__(256) prolongate_add_kernel(TransferArgs<CN, FN> a) {
  constexpr int KC = prolongate_components<P, NC>();
  __shared__ double lds[prolongate_lds<P, KC>()];
  const int cell = a.cell_begin + blockIdx.x;
  if (cell < a.cell_end) prolongate_cell<P, NC, CN, FN, KC>(a, cell, lds);
}
template <int P, int NC, typename CN, typename FN>
__global__ void __launch_bounds__(256) restrict_add_kernel(TransferArgs<CN, FN> a) {
  constexpr int KC = transfer_components<P, NC>();
  __shared__ double lds[transfer_lds<P, KC>()];
  const int cell = a.cell_begin + blockIdx.x;
  if (cell < a.cell_end) restrict_cell<P, NC, CN, FN, KC>(a, cell, lds);
}
template <int P, int NC, typename CN, typename FN>
__global__ void __launch_bounds__(256) interpolate_kernel(TransferArgs<CN, FN> a) {
  __shared__ double lds[transfer_lds<P>()];
  const int cell = a.cell_begin + blockIdx.x;
  if (cell < a.cell_end) interpolate_cell<P, NC, CN, FN>(a, cell, lds);
}

// Restriction in two launches instead of a fill and one per coarse colour: all
// coarse cells store their parts, then every coarse node sums them in colour
// order, rounding to CN after each as the colour launches do, so the result is
// theirs bit for bit.  The colour launches of a hierarchy's small levels hold a
// few cells each and take 5 to 13 us apiece whatever their size.
template <int P, int NC, typename CN, typename FN>
__global__ void __launch_bounds__(256) restrict_to_cells_kernel(TransferArgs<CN, FN> a) {
  constexpr int KC = transfer_components<P, NC>();
  __shared__ double lds[transfer_lds<P, KC>()];
  restrict_cell<P, NC, CN, FN, KC, true>(a, a.cell_begin + blockIdx.x, lds);
}

// coarse = the sums (0 on constrained components)
template <typename CN, int NC>
__global__ void __launch_bounds__(kGatherThreads)
    restrict_sums_kernel(GatherTables<double> g, CN *__restrict__ coarse, int64_t n_nodes) {
  const int64_t node = (int64_t)blockIdx.x * kGatherThreads + threadIdx.x;
  if (node >= n_nodes) return;
  const int b = g.offsets[node], e = g.offsets[node + 1];
  const unsigned m = g.cmask[node];
  CN acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = CN(0);
  for (int k = b; k < e; k += 4) {
    NodeValues<double, NC> v[4];
    uint32_t at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) at[u] = g.index && k + u < e ? g.index[k + u] : (uint32_t)(k + u);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < e) v[u] = load_node<double, NC>(g.contrib + (int64_t)at[u] * NC);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < e)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = (CN)((double)acc[c] + v[u].v[c]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if ((m >> c) & 1u) acc[c] = CN(0);
  store_node<CN, NC>(coarse + node * NC, acc);
}

}  // namespace mfg
