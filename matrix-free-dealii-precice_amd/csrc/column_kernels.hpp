// Sum-factorisation cell kernels with one thread per z column of a cell.
//
// The point-per-thread kernel (cell_kernels.hpp) reads 5 values and 5 matrix
// entries from LDS for every 5-term contraction and crosses 8 barriers per
// cell.  Here a thread owns the N nodes, and the N quadrature points, over one
// (i, j) of its cell, and a workgroup is one wave holding 64 / N^2 cells:
//  - z contractions stay in registers, with the 1D matrices as scalar operands;
//  - x and y contractions read lines from LDS, with the thread's two matrix
//    rows in registers for all N planes and components;
//  - the lanes of one wave execute LDS operations in order, so no barrier is
//    needed and each phase overwrites the tile the phase before has read;
//  - a thread's N point fields and nodes are N independent loads in flight.
// Every contraction sums the same terms in the same order as the
// point-per-thread kernel, so results are the same bit for bit and either may
// serve any launch.
//
// The price is registers: a thread holds its N values, z sums and scales, 90
// to 230 VGPRs in all (1 to 4 waves per SIMD), so a launch needs more cells to
// fill the GPU.  The next point's fields are loaded a whole point ahead and the
// two matrix rows stay in registers over the column: at 2 waves per SIMD both
// are worth more than a third wave (Q4 solid FP64 0.48 against 0.53 ms without
// them; bounding the registers instead spills, 0.69 ms and more).
//
// Measured, point per thread -> column per thread (vmult, colour launches,
// cubes of about 20M unknowns): heat Q4 FP64 606 -> 452 us, FP32 350 -> 277;
// Q5 640 -> 524, 424 -> 290; Q6 745 -> 431, 436 -> 267 (before the pins below); Q2 FP32 545 -> 454;
// solid (10 words) Q6 FP64 881 -> 577, FP32 341 -> 281; Q5 560 -> 518,
// 345 -> 313.  Solid Q4 and below are bound by the gather and scatter of the
// colour launches either way (Q4 FP64 480 and 481 us, FP32 264 and 288).
//
// Quadrature operator and references as in cell_kernels.hpp.
#pragma once
#include "cell_kernels.hpp"

namespace mfg {

template <int P>
constexpr int column_cells() {
  return 64 / ((P + 1) * (P + 1));
}

// whether there is a column kernel for the heat operator
template <int P, typename Number>
constexpr bool has_heat_columns() {
  return P >= 2 || sizeof(Number) == 4;
}
// whether there is a column kernel for the solid operators of a formulation
template <int P, typename Number>
constexpr bool has_solid_columns(bool formulation1) {
  return (P == 6 && sizeof(Number) == 8) || (P >= 5 && formulation1);
}
// Whether a launch of the heat operator on affine cells or of a tensor2 solid
// operator over n_cells cells (waves: workgroups of the column kernel) takes the
// column kernels; the results are the same bit for bit.  They hold 64 / (p+1)^2
// cells per wave at 1 to 4 waves per SIMD, so they need that many waves to fill
// the 1024 SIMDs; with fewer, the point-per-thread kernels spread the same
// cells over more waves.
// Measured over cubes of 2e4 to 2e7 unknowns, in one launch (GATHER) and in 8
// colours, times as point -> column in us:
//  - heat on affine cells: equal at about 600 waves (Q4 7.8 -> 9.2 at 172, Q2
//    8.4 -> 8.4 at 392), 7 to 50 % faster from 1000 (Q4 16.6 -> 14.8 at 1688,
//    Q6 16.8 -> 15.0 at 1000).  FP64 Q1 to Q3 is bound by its vector traffic
//    once that leaves the caches, from about 2^19 nodes a colour launch on: Q2
//    197 -> 185 at 64,000 cells a launch but 906 -> 943 at 314,432, Q3 133 ->
//    131 at 17,576 but 158 -> 169 at 21,952 and 293 -> 315 at 46,656 (one launch
//    over as many: 25.9 -> 28.8 and 46.5 -> 50.7); Q1 gains nothing at any size.
//  - solid Q6 FP64: 175 -> 146 at 614 waves, 881 -> 577 at 3724 (formulation 0
//    213 -> 176 and 1027 -> 743).
//  - solid Q5 and Q6 FP32, Q5 FP64, formulation 1: slower at 614 to 1000 waves
//    (Q6 FP32 91 -> 118, Q5 FP64 113.6 -> 114), faster at 1728 and above (Q6
//    FP32 36.6 -> 30.7, Q5 FP64 48.5 -> 45.9 at 2744).
//  - solid up to Q4: not faster at the large sizes.
template <int P, typename Number>
inline bool columns_pay(bool heat, bool formulation1, int n_cells, int waves) {
  constexpr bool fp64 = sizeof(Number) == 8;
  if (heat)
    return has_heat_columns<P, Number>() && waves >= 768 && !(fp64 && P <= 3 && n_cells > (1 << 19) / (P * P * P));
  return has_solid_columns<P, Number>(formulation1) && waves >= (fp64 && P == 6 ? 512 : 1536);
}

// LDS values of one cell: 2 NC N^3 (the point values or x gradients, and the y
// gradients), padded so that the lines which the cells of a wave read together
// start in different banks: the stride is 5, 9 and 17 modulo 32 values for
// N = 2, 3, 4 (without it the 4 cells of N = 4 met in the same banks).
template <int P, int NC>
constexpr int column_stride() {
  constexpr int N = P + 1, n = 2 * NC * N * N * N, want = N == 2 ? 5 : N == 3 ? 9 : 17;
  return N > 4 ? n : n + (want - n % 32 + 32) % 32;
}
// LDS values of a workgroup: the two 1D matrices and the cells
template <int P, int NC>
constexpr int column_lds() {
  return 2 * (P + 1) * (P + 1) + column_cells<P>() * column_stride<P, NC>();
}

// Orders the LDS accesses of the one wave of a workgroup; no instruction.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Completes x here and keeps the LDS loads that follow after it; no instruction.
template <typename Number>
__device__ inline void pin(Number &x) {
  asm volatile("" : "+v"(x) : : "memory");
}
// Whether each line's sum is completed before the loads of the next one.  The
// compiler otherwise gathers the loads of many lines first.  For the long lines
// of one component that costs waves (heat FP64 Q5 129 -> 121 VGPRs, 3 -> 4
// waves per SIMD: 650 -> 576 us at 24.6M unknowns, FP32 354 -> 336; Q6 546 ->
// 536, 344 -> 316); with three components, whose points have work enough
// between the loads, the loads in flight are worth more (solid Q6 FP64 727 us,
// pinned 861), and lines of 5 and less measured the same or 2% slower pinned.
template <int P, int NC>
constexpr bool pin_lines() {
  return NC == 1 && P >= 5;
}

// The cells [cell_begin, min(cell_begin + column_cells<P>(), cell_end)) on one
// wave.  assign, kToCells: as for cell_group.
template <int P, typename Number, class QOp, bool kToCells>
__device__ inline void cell_columns(const QOp &qop, const uint32_t *__restrict__ cell_nodes,
                                    const Number *__restrict__ src, Number *__restrict__ dst, int cell_begin,
                                    int cell_end, int assign, const Number *__restrict__ g_shape,
                                    const Number *__restrict__ g_colloc, Number *lds,
                                    const uint32_t *__restrict__ slots = nullptr) {
  constexpr int N = P + 1, NL = N * N, N3 = NL * N, NC = QOp::NC;
  Number *s_shape = lds, *s_colloc = lds + NL;
  const int t = threadIdx.x;
  for (int x = t; x < NL; x += 64) {
    s_shape[x] = g_shape[x];
    s_colloc[x] = g_colloc[x];
  }
  const int lc = t / NL, l = t - lc * NL, i = l % N, j = l / N;
  const int cell = cell_begin + lc;
  wave_lds_fence();
  if (lc >= column_cells<P>() || cell >= cell_end) return;
  Number *tile = lds + 2 * NL + lc * column_stride<P, NC>();
  Number *own = tile + l;                              // own[(c N + k) NL]: this thread's entries
  const Number *xl = tile + N * j, *yl = tile + i;     // its x lines (+ a) and y lines (+ a N)
  constexpr int B = NC * N3;                           // second half of the tile
  const ConstantPtr<Number> cS = as_constant(g_shape), cD = as_constant(g_colloc);
  // point k of the column: qb + lo + k NL, qb the same on every lane
  const int64_t qb = (int64_t)cell_begin * N3;
  const uint32_t lo = (uint32_t)(lc * N3 + l);

  uint32_t entry[N];
#pragma unroll
  for (int k = 0; k < N; ++k) entry[k] = (cell_nodes + qb)[lo + k * NL];
  const typename QOp::Cell cd = qop.load_cell(cell);
  Number v[NC][N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const NodeValues<Number, NC> u = load_node<Number, NC>(src + (int64_t)(entry[k] & kNodeMaskDev) * NC);
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c][k] = ((entry[k] >> (kConstraintShift + c)) & 1u) ? Number(0) : u.v[c];
  }
  typename QOp::Data qd = qop.load(qb, lo, l);

  Number ri[N], rj[N];  // the thread's rows (or columns) of the 1D matrix for x and y lines
  auto put = [&](int half) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int k = 0; k < N; ++k) own[half + (c * N + k) * NL] = v[c][k];
    wave_lds_fence();
  };
  // values at the points: x, y through LDS, z in registers
#pragma unroll
  for (int a = 0; a < N; ++a) {
    ri[a] = s_shape[i * N + a];
    rj[a] = s_shape[j * N + a];
  }
  put(0);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number r = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r += ri[a] * xl[(c * N + k) * NL + a];
      if constexpr (pin_lines<P, NC>()) pin(r);
      v[c][k] = r;
    }
  wave_lds_fence();
  put(0);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number r = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r += rj[a] * yl[(c * N + k) * NL + a * N];
      if constexpr (pin_lines<P, NC>()) pin(r);
      v[c][k] = r;
    }
  wave_lds_fence();
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    Number w[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number r = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r += cS[k * N + a] * v[c][a];
      w[k] = r;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) v[c][k] = w[k];
  }
#pragma unroll
  for (int a = 0; a < N; ++a) {
    ri[a] = s_colloc[i * N + a];
    rj[a] = s_colloc[j * N + a];
  }
  put(0);
  // point by point along the column: gradient, quadrature operation, and the
  // submitted gradients back to the tile (x in place of the plane's values,
  // which this plane's lanes have all read; y to the second half); the z part
  // of the transposed derivative is summed in registers
  Number z[NC][N], scale[N];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) z[c][k] = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    typename QOp::Data qn{};
    if (k + 1 < N) qn = qop.load(qb, lo + (k + 1) * NL, l + (k + 1) * NL);
    Number grad[NC][3];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      Number gx = 0, gy = 0, gz = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) gx += ri[a] * xl[(c * N + k) * NL + a];
#pragma unroll
      for (int a = 0; a < N; ++a) gy += rj[a] * yl[(c * N + k) * NL + a * N];
#pragma unroll
      for (int a = 0; a < N; ++a) gz += cD[k * N + a] * v[c][a];
      grad[c][0] = gx;
      grad[c][1] = gy;
      grad[c][2] = gz;
      if constexpr (pin_lines<P, NC>())
        asm volatile("" : "+v"(grad[c][0]), "+v"(grad[c][1]), "+v"(grad[c][2]) : : "memory");
    }
    wave_lds_fence();
    qop.apply_grad(cd, qd, grad);
    scale[k] = qop.value_scale(cd, qd);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      own[(c * N + k) * NL] = grad[c][0];
      own[B + (c * N + k) * NL] = grad[c][1];
#pragma unroll
      for (int a = 0; a < N; ++a) z[c][a] += cD[k * N + a] * grad[c][2];
    }
    __builtin_amdgcn_sched_barrier(0);
    qd = qn;
  }
  wave_lds_fence();
#pragma unroll
  for (int a = 0; a < N; ++a) {
    ri[a] = s_colloc[a * N + i];
    rj[a] = s_colloc[a * N + j];
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number rx = 0, ry = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) rx += ri[a] * xl[(c * N + k) * NL + a];
#pragma unroll
      for (int a = 0; a < N; ++a) ry += rj[a] * yl[B + (c * N + k) * NL + a * N];
      const Number s = scale[k] * v[c][k];
      v[c][k] = s + rx + ry + z[c][k];
      if constexpr (pin_lines<P, NC>()) pin(v[c][k]);
    }
  wave_lds_fence();
  // back to the nodes: z in registers, y, x through LDS
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    Number w[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number r = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r += cS[a * N + k] * v[c][a];
      w[k] = r;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) v[c][k] = w[k];
  }
#pragma unroll
  for (int a = 0; a < N; ++a) {
    ri[a] = s_shape[a * N + i];
    rj[a] = s_shape[a * N + j];
  }
  put(0);
  // dst of the thread's nodes (or the slots of its contributions), read while
  // the last two contractions run; the first colour touching a node stores
  // without reading
  Number dold[kToCells ? 1 : N][NC];
  uint32_t slot[kToCells ? N : 1];
  if constexpr (kToCells) {
#pragma unroll
    for (int k = 0; k < N; ++k) slot[k] = slots ? (slots + qb)[lo + k * NL] : (uint32_t)(qb + lo + k * NL);
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const bool first = assign && (entry[k] >> 31);
      const NodeValues<Number, NC> o =
          first ? NodeValues<Number, NC>{} : load_node<Number, NC>(dst + (int64_t)(entry[k] & kNodeMaskDev) * NC);
#pragma unroll
      for (int c = 0; c < NC; ++c) dold[k][c] = o.v[c];
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      Number r = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r += rj[a] * yl[(c * N + k) * NL + a * N];
      if constexpr (pin_lines<P, NC>()) pin(r);
      v[c][k] = r;
    }
  wave_lds_fence();
  put(0);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    Number r[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      r[c] = 0;
#pragma unroll
      for (int a = 0; a < N; ++a) r[c] += ri[a] * xl[(c * N + k) * NL + a];
    }
    if constexpr (kToCells) {
      store_node<Number, NC>(dst + (int64_t)slot[k] * NC, r);
    } else {
      Number *out = dst + (int64_t)(entry[k] & kNodeMaskDev) * NC;
#pragma unroll
      for (int c = 0; c < NC; ++c) r[c] = dold[k][c] + r[c];
      if (((entry[k] >> kConstraintShift) & ((1u << NC) - 1u)) == 0u) {
        store_node<Number, NC>(out, r);  // no constrained component: one wide store
      } else {
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (!((entry[k] >> (kConstraintShift + c)) & 1u)) out[c] = r[c];
      }
    }
  }
}

template <int P, typename Number, class QOp>
__global__ void __launch_bounds__(64) apply_columns(ApplyArgs<Number> a, QOp qop, int assign) {
  __shared__ Number lds[column_lds<P, QOp::NC>()];
  const int first_cell = a.cell_begin + xcd_remap(blockIdx.x, gridDim.x) * column_cells<P>();
  cell_columns<P, Number, QOp, false>(qop, a.cell_nodes, a.src, a.dst, first_cell, a.cell_end, assign, a.shape,
                                      a.colloc, lds);
  // rows of constrained dofs, as in apply_cells
  if (a.fix_mode) {
    const int64_t g = (int64_t)blockIdx.x * 64 + threadIdx.x;
    for (int64_t idx = g; idx < a.n_constrained; idx += (int64_t)gridDim.x * 64) {
      const int64_t dof = a.constrained[idx];
      if (a.fix_mode == 1) a.dst[dof] = a.src[dof];
      else a.dst[dof] += a.src[dof];
    }
  }
}

// GATHER schedule, first launch: as apply_cells_to_cells
template <int P, typename Number, class QOp>
__global__ void __launch_bounds__(64)
    apply_columns_to_cells(ApplyArgs<Number> a, QOp qop, Number *contrib) {
  __shared__ Number lds[column_lds<P, QOp::NC>()];
  const int first_cell = a.cell_begin + xcd_remap(blockIdx.x, gridDim.x) * column_cells<P>();
  cell_columns<P, Number, QOp, true>(qop, a.cell_nodes, a.src, contrib, first_cell, a.cell_end, 1, a.shape, a.colloc,
                                     lds, a.slots);
}

}  // namespace mfg
