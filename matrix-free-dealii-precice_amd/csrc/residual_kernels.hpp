// Newton residual (Solid::assemble_residual, fast FEEvaluation path,
// mf_elasticity.h:1764-1846): R = -int tau F^{-T} : Grad w dX
// + int rho (b - a) . w dX, on the reference configuration (MappingQ1).
#pragma once
#include "setup_kernels.hpp"
#include "vector_kernels.hpp"

namespace mfg {

template <typename Number>
struct ResidualArgs {
  const uint32_t *cell_nodes;
  int cell_begin, cell_end;
  const Number *u, *acc;
  Number *R;              // or (GATHER) the contribution buffer
  const uint32_t *slots;  // GATHER: places of the contributions
  const double *vertices;
  const Number *shape, *colloc;
  const double *points, *weights;
  Number mu, lambda, kappa, c_1, rho;
  Number body[3];
  int *error;
};

// Affine cells, formulation 1.  With H = Grad_X u, F = I + H:
//   tau F^{-T} = mu F - (mu - 2 lambda ln J) F^{-T}
//              = mu (H + (F^{-1} H)^T) + 2 lambda ln J F^{-T},
// since I - F^{-1} = F^{-1} H, and J - 1 = tr H + the second minors + det H.
// No term cancels down from the size of the identity to that of the strain
// (mu b - s I does), and b and tau are not formed.
template <typename Number>
__device__ inline bool residual_point_affine(const ResidualArgs<Number> &a, ConstantPtr<double> X, double wq,
                                             const Number (&gr)[3][3], const Number (&av)[3], Number (&val)[3],
                                             Number (&grad)[3][3]) {
  double Jr[3][3], R[3][3];
  affine_jacobian(X, Jr);
  inv3(Jr, R);
  const double w = fabs(det3(Jr)) * wq;
  Number H[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int e = 0; e < 3; ++e) H[d][e] = gr[d][0] * R[0][e] + gr[d][1] * R[1][e] + gr[d][2] * R[2][e];
  const Number Jm1 = (H[0][0] + H[1][1] + H[2][2]) + (H[0][0] * H[1][1] - H[0][1] * H[1][0]) +
                     (H[0][0] * H[2][2] - H[0][2] * H[2][0]) + (H[1][1] * H[2][2] - H[1][2] * H[2][1]) + det3(H);
  Number Fi[3][3];
  {
    Number F[3][3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int e = 0; e < 3; ++e) F[d][e] = H[d][e] + (d == e ? Number(1) : Number(0));
    inv3(F, Fi);
  }
  const Number l = Number(2) * a.lambda * log1p(Jm1);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    Number Pc[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const Number FiH = Fi[e][0] * H[0][c] + Fi[e][1] * H[1][c] + Fi[e][2] * H[2][c];
      Pc[e] = a.mu * (H[c][e] + FiH) + l * Fi[e][c];
    }
#pragma unroll
    for (int f = 0; f < 3; ++f) grad[c][f] = -w * (Pc[0] * R[f][0] + Pc[1] * R[f][1] + Pc[2] * R[f][2]);
    val[c] = w * a.rho * (a.body[c] - av[c]);
  }
  return Jm1 > Number(-1);
}

// Any cell and formulation.
template <typename Number>
__device__ inline bool residual_point(const ResidualArgs<Number> &a, int formulation, const double (&Jr)[3][3],
                                      double wq, const Number (&gr)[3][3], const Number (&av)[3], Number (&val)[3],
                                      Number (&grad)[3][3]) {
  double Jri[3][3];
  inv3(Jr, Jri);
  const Number jxw = (Number)(fabs(det3(Jr)) * wq);
  Number F[3][3], Fi[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int e = 0; e < 3; ++e)
      F[d][e] = gr[d][0] * (Number)Jri[0][e] + gr[d][1] * (Number)Jri[1][e] + gr[d][2] * (Number)Jri[2][e] +
                (d == e ? Number(1) : Number(0));
  const Number J = det3(F);
  inv3(F, Fi);
  Number b[3][3], tau[3][3];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) b[x][y] = F[x][0] * F[y][0] + F[x][1] * F[y][1] + F[x][2] * F[y][2];
  if (formulation == 1) {  // material.h:148-158
    const Number tmp = a.mu - Number(2) * a.lambda * log(J);
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y) tau[x][y] = a.mu * b[x][y] - (x == y ? tmp : Number(0));
  } else {  // material.h:125-147
    const Number Jm23 = pow(J, Number(-2.0 / 3.0));
    const Number dpsi = (a.kappa / Number(2)) * (J - Number(1) / J);
    const Number tr = Number(2) * a.c_1 * Jm23 * (b[0][0] + b[1][1] + b[2][2]);
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y)
        tau[x][y] = Number(2) * a.c_1 * Jm23 * b[x][y] + (x == y ? dpsi * J - tr / Number(3) : Number(0));
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    Number Pd[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) Pd[e] = -(tau[d][0] * Fi[e][0] + tau[d][1] * Fi[e][1] + tau[d][2] * Fi[e][2]);
#pragma unroll
    for (int f = 0; f < 3; ++f)
      grad[d][f] = jxw * (Pd[0] * (Number)Jri[f][0] + Pd[1] * (Number)Jri[f][1] + Pd[2] * (Number)Jri[f][2]);
    val[d] = jxw * a.rho * (a.body[d] - av[d]);
  }
  return J > Number(0);
}

// KIND 0: affine cells, formulation 1; 1, 2: any cell, formulation 1 or 0.  u
// and the acceleration go through the value sweeps together (12 tile slots, 8
// barriers per cell); the 1D matrices and both fields are loaded before the
// first barrier.  The first colour that touches a node stores (0 on constrained
// components), which makes a zero fill unnecessary; kToCells: the contributions
// of the GATHER schedule.
// Measured with the norm read back into pinned memory, against two cells per
// workgroup, a fill, colour launches at every size, the per-point trilinear
// Jacobian, b and tau: Q4 64x16x16 cells 212 -> 162 us, Q3 cubes of 20K, 0.3M
// and 3M unknowns 117 -> 28, 124 -> 40, 224 -> 149 us; Q6 155 -> 33, 159 -> 46,
// 272 -> 236.  Bounding the registers to 4 waves per SIMD instead of 3 (12 to
// 30 spilled) was not faster at any degree.
template <int P, int CPB, int KIND, bool kToCells, typename Number>
__global__ void __launch_bounds__((block_threads<P, CPB>())) residual_cells(ResidualArgs<Number> a) {
  constexpr int N = P + 1, N3 = N * N * N, NL = N * N;
  __shared__ Number s_shape[NL], s_colloc[NL];
  __shared__ Number s_tile[CPB * 12 * N3];
  const int t = threadIdx.x;
  const int lc_raw = t / N3;
  const bool pad = lc_raw >= CPB;
  const int lc = pad ? CPB - 1 : lc_raw;
  const int pt = pad ? 0 : t - lc_raw * N3;
  Tile<N, Number> T;
  T.base = s_tile + lc * 12 * N3;
  T.pt = pt;
  T.i = pt % N;
  T.j = (pt / N) % N;
  T.k = pt / NL;
  T.writer = !pad;
  const int first_cell = a.cell_begin + xcd_remap(blockIdx.x, gridDim.x) * CPB, cell = first_cell + lc;
  const bool active = !pad && cell < a.cell_end;
  const int64_t qb = (int64_t)first_cell * N3;
  const uint32_t lo = active ? (uint32_t)t : 0u;
  const uint32_t entry = active ? (a.cell_nodes + qb)[lo] : 0u;
  uint32_t slot = 0;
  if constexpr (kToCells) slot = a.slots ? (a.slots + qb)[lo] : (uint32_t)(qb + lo);
  Number sh = 0, co = 0;
  if (t < NL) {
    sh = a.shape[t];
    co = a.colloc[t];
  }
  const int64_t node = entry & kNodeMaskDev;
  Number v[6];  // u, acc: read_dof_values_plain
  {
    const NodeValues<Number, 3> x = active ? load_node<Number, 3>(a.u + node * 3) : NodeValues<Number, 3>{};
    const NodeValues<Number, 3> y = active ? load_node<Number, 3>(a.acc + node * 3) : NodeValues<Number, 3>{};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      v[c] = x.v[c];
      v[3 + c] = y.v[c];
    }
  }
  const bool first = entry >> 31;
  NodeValues<Number, 3> old{};
  if constexpr (!kToCells)
    if (active && !first) old = load_node<Number, 3>(a.R + node * 3);
  if (t < NL) {  // published by the first barrier
    s_shape[t] = sh;
    s_colloc[t] = co;
  }
  // values at the points: slots 0..5 -> 6..11 -> 0..5 -> registers
#pragma unroll
  for (int c = 0; c < 6; ++c) T.put(c, v[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 6; ++c) v[c] = T.template line<0>(s_shape, T.i, c);
#pragma unroll
  for (int c = 0; c < 6; ++c) T.put(6 + c, v[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 6; ++c) v[c] = T.template line<1>(s_shape, T.j, 6 + c);
#pragma unroll
  for (int c = 0; c < 6; ++c) T.put(c, v[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 6; ++c) v[c] = T.template line<2>(s_shape, T.k, c);
  // slots 6..8 (last read before the barrier above): the values of u
#pragma unroll
  for (int c = 0; c < 3; ++c) T.put(6 + c, v[c]);
  __syncthreads();
  Number gr[3][3], av[3] = {v[3], v[4], v[5]}, val[3], grad[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    gr[c][0] = T.template line<0>(s_colloc, T.i, 6 + c);
    gr[c][1] = T.template line<1>(s_colloc, T.j, 6 + c);
    gr[c][2] = T.template line<2>(s_colloc, T.k, 6 + c);
  }
  const double wq = a.weights[T.i] * a.weights[T.j] * a.weights[T.k];
  const int vcell = CPB == 1 ? __builtin_amdgcn_readfirstlane(first_cell) : active ? cell : first_cell;
  const ConstantPtr<double> X = as_constant(a.vertices) + (int64_t)vcell * 24;
  bool ok;
  if constexpr (KIND == 0) {
    ok = residual_point_affine(a, X, wq, gr, av, val, grad);
  } else {
    double Jr[3][3];
    trilinear_jacobian(X, a.points[T.i], a.points[T.j], a.points[T.k], Jr);
    ok = residual_point(a, KIND == 1 ? 1 : 0, Jr, wq, gr, av, val, grad);
  }
  if (active && !ok) *a.error = 1;
  // back to the nodes: the gradients in slots 0..5 and 9..11, which no line
  // since the last barrier reads
  auto g_slot = [](int x) { return x < 6 ? x : x + 3; };
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int f = 0; f < 3; ++f) T.put(g_slot(3 * c + f), grad[c][f]);
  __syncthreads();
  // Colour launches: each component's sum is completed before the loads of the
  // next one.  Without it the loads of all 9 lines come first, at 138 (Q4) and
  // 156 VGPRs (Q6), 3 waves per SIMD; with it 104 each, 4 waves.  3M
  // unknowns: Q4 164 -> 159 us, Q5 168 -> 169, Q6 241 -> 221.  Below Q4 and in
  // the GATHER form the loads in flight are worth more (Q3 147 -> 153, Q2 198
  // -> 204; GATHER 1% slower), as they are in the forward lines of any degree.
  constexpr bool kPin = P >= 4 && !kToCells;
  Number r[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    r[c] = val[c] + T.template line_t<0>(s_colloc, T.i, g_slot(3 * c + 0)) +
           T.template line_t<1>(s_colloc, T.j, g_slot(3 * c + 1)) +
           T.template line_t<2>(s_colloc, T.k, g_slot(3 * c + 2));
    if constexpr (kPin) asm volatile("" : "+v"(r[c]) : : "memory");
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) T.put(6 + c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = T.template line_t<2>(s_shape, T.k, 6 + c);
#pragma unroll
  for (int c = 0; c < 3; ++c) T.put(c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = T.template line_t<1>(s_shape, T.j, c);
#pragma unroll
  for (int c = 0; c < 3; ++c) T.put(6 + c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = T.template line_t<0>(s_shape, T.i, 6 + c);
  if (!active) return;
  if constexpr (kToCells) {
    store_node<Number, 3>(a.R + (int64_t)slot * 3, r);
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) r[c] = (entry >> (kConstraintShift + c)) & 1u ? Number(0) : old.v[c] + r[c];
    store_node<Number, 3>(a.R + node * 3, r);
  }
}

// R = the nodes' sums, 0 on constrained components
template <typename Number>
__global__ void __launch_bounds__(kGatherThreads)
    residual_sums_kernel(GatherTables<Number> g, Number *__restrict__ R, int64_t n_nodes) {
  const int64_t node = (int64_t)blockIdx.x * kGatherThreads + threadIdx.x;
  if (node >= n_nodes) return;
  const unsigned m = g.cmask[node];
  Number t[3] = {};
  add_contributions<Number, 3>(g.contrib, g.index, g.offsets[node], g.offsets[node + 1], t);
#pragma unroll
  for (int c = 0; c < 3; ++c)
    if ((m >> c) & 1u) t[c] = 0;
  store_node<Number, 3>(R + node * 3, t);
}

// Newmark: a = a1 du - a2 v_old - a3 a_old (update_acceleration, :1614-1620)
template <typename T>
__global__ void newmark_acc_kernel(T *acc, const T *du, const T *v_old, const T *a_old, double a1, double a2,
                                   double a3, int64_t n) {
  MFG_GRID_STRIDE(i, n) acc[i] = (T)(a1 * (double)du[i] - a2 * (double)v_old[i] - a3 * (double)a_old[i]);
}
// v = a4 du + a5 v_old + a6 a_old (update_velocity, :1600-1609)
template <typename T>
__global__ void newmark_vel_kernel(T *vel, const T *du, const T *v_old, const T *a_old, double a4, double a5,
                                   double a6, int64_t n) {
  MFG_GRID_STRIDE(i, n) vel[i] = (T)(a4 * (double)du[i] + a5 * (double)v_old[i] + a6 * (double)a_old[i]);
}
// x += y ; z += y
template <typename T>
__global__ void add2_kernel(T *x, T *z, const T *y, int64_t n) {
  MFG_GRID_STRIDE(i, n) {
    x[i] += y[i];
    z[i] += y[i];
  }
}

}  // namespace mfg
