// Per-linearisation set-up kernels: the quadrature cache (NeoHookOperator::
// cache, mf_nh_operator.h:392-523, with the deformed-frame geometry that
// MappingQEulerian provides to the tensor2 caching, mf_elasticity.h:951-952)
// and the operator diagonal (compute_diagonal, :1023-1060).
#pragma once
#include "cell_kernels.hpp"

namespace mfg {

template <typename Number>
struct CacheArgs {
  const uint32_t *cell_nodes;
  int cell_begin, cell_end;  // stored cells of one material
  const void *u;     // displacement, precision u_fp32 ? float : double
  int u_fp32;
  const double *vertices;  // 24 per stored cell
  const Number *shape, *colloc;
  const double *points, *weights;  // Gauss rule on [0,1], N each
  Number *qd;
  int64_t nqp;
  Number mu, lambda;
  int formulation;
  int caching;  // MFG_CACHING_*
  int jxw_ref_field;  // tensor2 formulation 1: store JxW_ref as field 16 (not supplied per cell)
  // tensor2 formulation 1, MFG_T2_GRADIENT: 1 stores the operator's 10 fields
  // (Jinv_cur, s), and the displacement itself to u_copy; 2 stores Grad_xi u
  // and s (what mfg_operator_qp_data exports) field by field in input cell order
  int t2_gradient;
  Number *u_copy;       // 3 per node, with t2_gradient 1
  const int32_t *perm;  // with t2_gradient 2: input index of every stored cell
  int *error;   // set to 1 if det F <= 0 anywhere (not with t2_gradient 2)
};

template <typename Number>
__device__ inline Number det3(const Number (&A)[3][3]) {
  return A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1]) - A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0]) +
         A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
}
template <typename Number>
__device__ inline void inv3(const Number (&A)[3][3], Number (&R)[3][3]) {
  const Number id = Number(1) / det3(A);
  R[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) * id;
  R[0][1] = (A[0][2] * A[2][1] - A[0][1] * A[2][2]) * id;
  R[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) * id;
  R[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) * id;
  R[1][1] = (A[0][0] * A[2][2] - A[0][2] * A[2][0]) * id;
  R[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) * id;
  R[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) * id;
  R[2][1] = (A[0][1] * A[2][0] - A[0][0] * A[2][1]) * id;
  R[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) * id;
}

// Trilinear Jacobian dX_e/dxi_f at reference point xi from 8 vertices.
template <class Ptr>
__device__ inline void trilinear_jacobian(Ptr v, double x0, double x1, double x2, double (&J)[3][3]) {
#pragma unroll
  for (int e = 0; e < 3; ++e)
#pragma unroll
    for (int f = 0; f < 3; ++f) J[e][f] = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int b0 = c & 1, b1 = (c >> 1) & 1, b2 = (c >> 2) & 1;
    const double n0 = b0 ? x0 : 1 - x0, n1 = b1 ? x1 : 1 - x1, n2 = b2 ? x2 : 1 - x2;
    const double d0 = b0 ? 1 : -1, d1 = b1 ? 1 : -1, d2 = b2 ? 1 : -1;
    const double g0 = d0 * n1 * n2, g1 = n0 * d1 * n2, g2 = n0 * n1 * d2;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const double X = v[c * 3 + e];
      J[e][0] += X * g0;
      J[e][1] += X * g1;
      J[e][2] += X * g2;
    }
  }
}

// The same on an affine cell, where it is constant: the edge differences, as
// the host forms the per-cell tables from them.  The general sum over the
// vertices cancels from the size of the coordinates down to that of the cell
// (1e-14 of the Jacobian on the 32-cell beam, 4 long); the differences do not.
template <class Ptr>
__device__ inline void affine_jacobian(Ptr v, double (&J)[3][3]) {
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    J[e][0] = v[3 + e] - v[e];
    J[e][1] = v[6 + e] - v[e];
    J[e][2] = v[12 + e] - v[e];
  }
}

// Workgroups: where N^3 is no multiple of 8, the fields of neighbouring cells
// share cache lines, and an XCD takes contiguous cells so that they meet in one
// L2; otherwise all XCDs walk the fields together.  15M unknowns FP64, contiguous
// / together: tensor2 words non-affine Q1 2001 / 1810 us, Q4 479 / 538, Q6 460 /
// 475; formulation 0 Q3 615 / 538; tensor4 (5M) Q4 406 / 447.
// kAffine: every cell's trilinear map is affine.  Both Jacobians in one kernel
// take Q1 and Q2 FP64 from 4 waves per SIMD to 3: 1.2M unknowns Q1 non-affine 206
// against 181 us (178 from the Jacobian of the vertices in point order alone),
// 1.5M Q2 105 against 95.  Q1 and Q2 FP64 are 2 registers above 4 waves' share;
// bounded to it, 3 spill (Q2).
// kStream: with t2_gradient 1, the fields are stored past the caches (a run-time
// choice is no use: the compiler merges the two stores into a plain one).
template <int P, int CPB, typename Number, bool kAffine, bool kStream = false>
__global__ void __launch_bounds__((block_threads<P, CPB>()), (P <= 2 && sizeof(Number) == 8 ? 4 : 1))
    cache_solid(CacheArgs<Number> a) {
  constexpr int N = P + 1, N3 = N * N * N;
  constexpr bool kNeighboursShareLines = N3 % 8 != 0;
  __shared__ Number s_shape[N * N], s_colloc[N * N];
  __shared__ Number s_tile[CPB * 6 * N3];
  const int t = threadIdx.x;
  const int lc_raw = t / N3;
  const bool pad = lc_raw >= CPB;
  const int lc = pad ? CPB - 1 : lc_raw;
  const int pt = pad ? 0 : t - lc_raw * N3;
  Tile<N, Number> T;
  T.base = s_tile + lc * 6 * N3;
  T.pt = pt;
  T.i = pt % N;
  T.j = (pt / N) % N;
  T.k = pt / (N * N);
  T.writer = !pad;
  const int block = kNeighboursShareLines ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int first_cell = a.cell_begin + block * CPB, cell = first_cell + lc;
  const bool active = !pad && cell < a.cell_end;
  const int64_t qidx = (int64_t)first_cell * N3 + (active ? t : 0);
  const uint32_t entry = active ? a.cell_nodes[qidx] : 0u;
  Number sh = 0, co = 0;
  if (t < N * N) {
    sh = a.shape[t];
    co = a.colloc[t];
  }
  const int64_t node = (int64_t)(entry & kNodeMaskDev);
  Number u[3];
  // read_dof_values_plain: constrained entries are read as stored
  if (a.u_fp32) {
    const NodeValues<float, 3> x = active ? load_node<float, 3>((const float *)a.u + node * 3) : NodeValues<float, 3>{};
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c] = (Number)x.v[c];
  } else {
    const NodeValues<double, 3> x =
        active ? load_node<double, 3>((const double *)a.u + node * 3) : NodeValues<double, 3>{};
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c] = (Number)x.v[c];
  }
  // one (cell, point) of every node carries the first-touch bit
  if (a.u_copy && active && (entry >> 31)) store_node<Number, 3>(a.u_copy + node * 3, u);
  if (t < N * N) {  // published by the first barrier of the sweeps
    s_shape[t] = sh;
    s_colloc[t] = co;
  }
  Number gr[3][3];
  evaluate_g<N, 3, Number, rolled_components<N, true>()>(T, s_shape, s_colloc, u, gr);
  if (!active) return;

  double Jr[3][3], Jri[3][3];
  auto jacobian = [&](auto X) {
    if constexpr (kAffine) affine_jacobian(X, Jr);
    else trilinear_jacobian(X, a.points[T.i], a.points[T.j], a.points[T.k], Jr);
  };
  // one cell per workgroup: the vertices come in as scalar loads
  if constexpr (CPB == 1)
    jacobian(as_constant(a.vertices) + (int64_t)__builtin_amdgcn_readfirstlane(first_cell) * 24);
  else
    jacobian(a.vertices + (int64_t)cell * 24);
  {
    const double id = 1.0 / (Jr[0][0] * (Jr[1][1] * Jr[2][2] - Jr[1][2] * Jr[2][1]) -
                             Jr[0][1] * (Jr[1][0] * Jr[2][2] - Jr[1][2] * Jr[2][0]) +
                             Jr[0][2] * (Jr[1][0] * Jr[2][1] - Jr[1][1] * Jr[2][0]));
    Jri[0][0] = (Jr[1][1] * Jr[2][2] - Jr[1][2] * Jr[2][1]) * id;
    Jri[0][1] = (Jr[0][2] * Jr[2][1] - Jr[0][1] * Jr[2][2]) * id;
    Jri[0][2] = (Jr[0][1] * Jr[1][2] - Jr[0][2] * Jr[1][1]) * id;
    Jri[1][0] = (Jr[1][2] * Jr[2][0] - Jr[1][0] * Jr[2][2]) * id;
    Jri[1][1] = (Jr[0][0] * Jr[2][2] - Jr[0][2] * Jr[2][0]) * id;
    Jri[1][2] = (Jr[0][2] * Jr[1][0] - Jr[0][0] * Jr[1][2]) * id;
    Jri[2][0] = (Jr[1][0] * Jr[2][1] - Jr[1][1] * Jr[2][0]) * id;
    Jri[2][1] = (Jr[0][1] * Jr[2][0] - Jr[0][0] * Jr[2][1]) * id;
    Jri[2][2] = (Jr[0][0] * Jr[1][1] - Jr[0][1] * Jr[1][0]) * id;
  }
  // F = I + Grad_X u ; current-frame Jacobian dx/dxi = dX/dxi + du/dxi
  Number F[3][3], Jc[3][3], Jci[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      F[d][e] = gr[d][0] * (Number)Jri[0][e] + gr[d][1] * (Number)Jri[1][e] + gr[d][2] * (Number)Jri[2][e] +
                (d == e ? Number(1) : Number(0));
      Jc[d][e] = (Number)Jr[d][e] + gr[d][e];
    }
  const Number J = det3(F);
  const int64_t n = a.nqp;
  if (a.t2_gradient == 2) {
    const int64_t at = (int64_t)a.perm[cell] * N3 + pt;
#pragma unroll
    for (int f = 0; f < 9; ++f) a.qd[f * n + at] = gr[f / 3][f % 3];
    a.qd[9 * n + at] = a.mu - Number(2) * a.lambda * log(J);
    return;
  }
  if (!(J > Number(0))) {
    *a.error = 1;
    return;
  }
  const double wq = a.weights[T.i] * a.weights[T.j] * a.weights[T.k];
  const Number scalar = a.mu - Number(2) * a.lambda * log(J);
  if (a.t2_gradient) {  // 9 words and s, in pairs of fields
    Number f10[10];
    inv3(Jc, Jci);
#pragma unroll
    for (int f = 0; f < 9; ++f) f10[f] = Jci[f / 3][f % 3];
    f10[9] = scalar;
    typedef Number Pair __attribute__((ext_vector_type(2)));
    Pair *qp = reinterpret_cast<Pair *>(a.qd);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const Pair x{f10[2 * k], f10[2 * k + 1]};
      if constexpr (kStream) __builtin_nontemporal_store(x, qp + k * n + qidx);
      else qp[k * n + qidx] = x;
    }
    return;
  }
  if (a.caching == MFG_CACHING_SCALAR_REFERENTIAL || a.caching == MFG_CACHING_TENSOR4_NS) {
    // reference-frame geometry (MappingQ1 of the reference configuration)
    const double detr = Jr[0][0] * (Jr[1][1] * Jr[2][2] - Jr[1][2] * Jr[2][1]) -
                        Jr[0][1] * (Jr[1][0] * Jr[2][2] - Jr[1][2] * Jr[2][0]) +
                        Jr[0][2] * (Jr[1][0] * Jr[2][1] - Jr[1][1] * Jr[2][0]);
#pragma unroll
    for (int f = 0; f < 9; ++f) a.qd[f * n + qidx] = (Number)Jri[f / 3][f % 3];
    a.qd[9 * n + qidx] = (Number)(wq * fabs(detr));
    if (a.caching == MFG_CACHING_SCALAR_REFERENTIAL) {  // mf_nh_operator.h:442-455
      a.qd[10 * n + qidx] = scalar;
      return;
    }
    // tensor4_ns (mf_nh_operator.h:495-516): 2 lambda F^-T (x) F^-T + s_c F^-T (x)_il F^-1 + mu I (x)_ik I
    Number Fi[3][3];
    inv3(F, Fi);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int l = 0; l < 3; ++l)
            a.qd[(10 + ((i * 3 + j) * 3 + k) * 3 + l) * n + qidx] =
                Number(2) * a.lambda * Fi[j][i] * Fi[l][k] + scalar * Fi[l][i] * Fi[j][k] +
                ((i == k && j == l) ? a.mu : Number(0));
    return;
  }
  inv3(Jc, Jci);
  const Number jxw = (Number)wq * fabs(det3(Jc));
  // tensor2, formulation 1 keeps its first 16 fields in pairs (see QSolidT2F1)
  const bool paired = a.formulation == 1 && a.caching == MFG_CACHING_TENSOR2;
  auto at = [&](int f) -> int64_t { return paired && f < 16 ? ((f >> 1) * n + qidx) * 2 + (f & 1) : f * n + qidx; };
#pragma unroll
  for (int f = 0; f < 9; ++f) a.qd[at(f)] = Jci[f / 3][f % 3];
  if (a.formulation == 0) {
    // mf_nh_operator.h:419-440: J^{-1/3} and F
    a.qd[9 * n + qidx] = jxw;
    a.qd[10 * n + qidx] = pow(J, Number(-1.0 / 3.0));
#pragma unroll
    for (int f = 0; f < 9; ++f) a.qd[(11 + f) * n + qidx] = F[f / 3][f % 3];
    return;
  }
  const Number invJ = Number(1) / J;
  Number b[3][3];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y) b[x][y] = F[x][0] * F[y][0] + F[x][1] * F[y][1] + F[x][2] * F[y][2];
  if (a.caching == MFG_CACHING_TENSOR4) {  // mf_nh_operator.h:478-494
    a.qd[9 * n + qidx] = jxw;
    a.qd[10 * n + qidx] = invJ;
#pragma unroll
    for (int s6 = 0; s6 < 6; ++s6) {
      const Number tau = a.mu * b[kSymI[s6]][kSymJ[s6]] - (kSymI[s6] == kSymJ[s6] ? scalar : Number(0));
      a.qd[(11 + s6) * n + qidx] = tau / J;
    }
    // C_ijkl = (2 s_c / J) (d_ik d_jl + d_il d_jk)/2 + (2 lambda / J) d_ij d_kl over symmetric pairs
#pragma unroll
    for (int s6 = 0; s6 < 6; ++s6)
#pragma unroll
      for (int t6 = 0; t6 < 6; ++t6) {
        const int i = kSymI[s6], j = kSymJ[s6], k = kSymI[t6], l = kSymJ[t6];
        const Number S = Number(0.5) * (Number((i == k && j == l) ? 1 : 0) + Number((i == l && j == k) ? 1 : 0));
        const Number IxI = (i == j && k == l) ? Number(1) : Number(0);
        a.qd[(17 + 6 * s6 + t6) * n + qidx] = (scalar * Number(2) / J) * S + (a.lambda * Number(2) / J) * IxI;
      }
    return;
  }
  // tensor2, formulation 1 (mf_nh_operator.h:456-477): the reference's
  // 2 s / J and tau / J times the current JxW = JxW_ref J, i.e. JxW_ref s and
  // JxW_ref tau, plus JxW_ref itself unless the operator takes it per cell
  const double detr = Jr[0][0] * (Jr[1][1] * Jr[2][2] - Jr[1][2] * Jr[2][1]) -
                      Jr[0][1] * (Jr[1][0] * Jr[2][2] - Jr[1][2] * Jr[2][0]) +
                      Jr[0][2] * (Jr[1][0] * Jr[2][1] - Jr[1][1] * Jr[2][0]);
  const Number jxw_ref = (Number)(wq * fabs(detr));
  a.qd[at(9)] = jxw_ref * scalar;
#pragma unroll
  for (int s6 = 0; s6 < 6; ++s6) {
    const Number tau = a.mu * b[kSymI[s6]][kSymJ[s6]] - (kSymI[s6] == kSymJ[s6] ? scalar : Number(0));
    a.qd[at(10 + s6)] = jxw_ref * tau;
  }
  if (a.jxw_ref_field) a.qd[at(16)] = jxw_ref;
}

// ---------------------------------------------------------- diagonal ---
// The diagonal entry of dof (node a, component d) is
//   sum_q [ m_d(q) phi_a(q)^2 + sum_{f,g} G_d[f][g](q) dphi_a/dxi_f dphi_a/dxi_g ],
// where m_d and G_d come from applying the quadrature op to unit values and
// unit reference gradients.  Each of the 7 terms (m; G_xx, G_yy, G_zz; G_xy,
// G_xz, G_yz with their transposes) is a tensor-product sum over q with squared
// 1D matrices (phi^2, phi*phi', phi'^2), evaluated with the same transposed
// sweeps as integrate.  After a direction's sweep the terms whose remaining
// directions take the same matrices are added: 7 lines along z, 6 along y, 3
// along x per component instead of 7 each.  Pinning each component's results
// before the next component's lines takes the FP64 kernel from 198 - 256 VGPRs
// to 66 - 82 (Q3 - Q6).  compute_diagonal(), against unit vectors through the
// quadrature op and a launch per colour: Q3 cubes FP64 of 20K, 0.3M and 3M
// unknowns 93 -> 17, 99 -> 29, 222 -> 160 us; Q6 220 -> 22, 237 -> 35, 690 ->
// 246; Q1 3M unknowns 1669 -> 268 us (8 cells per workgroup instead of one).

// the 7 terms of every component at a point
template <class QOp>
struct DiagonalTerms {
  template <typename Number>
  static __device__ void eval(const QOp &qop, const typename QOp::Cell &cd, const typename QOp::Data &qd,
                              Number (&coef)[7 * QOp::NC]) {
    constexpr int NC = QOp::NC;
    const Number m = qop.value_scale(cd, qd);
#pragma unroll
    for (int d = 0; d < NC; ++d) {
      Number G[3][3];
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        Number g[NC][3] = {};
        g[d][h] = 1;
        qop.apply_grad(cd, qd, g);
#pragma unroll
        for (int f = 0; f < 3; ++f) G[f][h] = g[d][f];
      }
      coef[d * 7] = m;
      coef[d * 7 + 1] = G[0][0];
      coef[d * 7 + 2] = G[1][1];
      coef[d * 7 + 3] = G[2][2];
      coef[d * 7 + 4] = G[0][1] + G[1][0];
      coef[d * 7 + 5] = G[0][2] + G[2][0];
      coef[d * 7 + 6] = G[1][2] + G[2][1];
    }
  }
};
// QSolidT2F1G: G_d = w (mu G + (s + 2 lambda) j_d j_d^T), j_d the column d of Jinv_cur
template <typename Number, bool kEarlyCell, bool kCartesian>
struct DiagonalTerms<QSolidT2F1G<Number, kEarlyCell, kCartesian>> {
  using QOp = QSolidT2F1G<Number, kEarlyCell, kCartesian>;
  static __device__ void eval(const QOp &qop, const typename QOp::Cell &cd, const typename QOp::Data &qd,
                              Number (&coef)[21]) {
    const Number m = qop.value_scale(cd, qd), w = cd.jxw * qd.w, wm = w * qop.mu, ws = w * (qd.s + qop.two_lambda);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const Number j0 = qd.ji[d], j1 = qd.ji[3 + d], j2 = qd.ji[6 + d];
      const Number s0 = ws * j0, s1 = ws * j1, s2 = ws * j2;
      coef[d * 7] = m;
      coef[d * 7 + 1] = wm * cd.g[0] + s0 * j0;
      coef[d * 7 + 2] = wm * cd.g[1] + s1 * j1;
      coef[d * 7 + 3] = wm * cd.g[2] + s2 * j2;
      const Number off[3] = {s0 * j1, s0 * j2, s1 * j2};
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        if constexpr (kCartesian) coef[d * 7 + 4 + x] = Number(2) * off[x];
        else coef[d * 7 + 4 + x] = Number(2) * (wm * cd.g[3 + x] + off[x]);
      }
    }
  }
};
// heat on affine cells: c dt JxW G
template <typename Number>
struct DiagonalTerms<QHeat<Number, true>> {
  using QOp = QHeat<Number, true>;
  static __device__ void eval(const QOp &qop, const typename QOp::Cell &cd, const typename QOp::Data &qd,
                              Number (&coef)[7]) {
    coef[0] = qop.value_scale(cd, qd);
    const Number s = qd.c * qop.dt * coef[0];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      coef[1 + x] = s * cd.g[x];
      coef[4 + x] = Number(2) * (s * cd.g[3 + x]);
    }
  }
};

template <typename Number>
struct DiagArgs {
  const uint32_t *cell_nodes;
  int cell_begin, cell_end;  // one colour: cells share no node; or (GATHER) all cells
  const Number *sq;  // 3 x N x N: SS, SD, DD
  const Number *shape, *colloc;  // for ops that read a nodal field
  Number *diag;                  // or (GATHER) the contribution buffer
  const uint32_t *slots;         // GATHER: places of the contributions
};

// The first colour touching a node stores; constrained components are left.
template <int P, int CPB, bool kToCells, typename Number, class QOp>
__global__ void __launch_bounds__((block_threads<P, CPB>())) diagonal_cells(DiagArgs<Number> a, QOp qop) {
  constexpr int N = P + 1, N3 = N * N * N, NC = QOp::NC, NTERM = 7 * NC;
  __shared__ Number s_sq[3 * N * N];
  __shared__ Number s_tile[CPB * NTERM * N3];
  const int t = threadIdx.x;
  for (int x = t; x < 3 * N * N; x += blockDim.x) s_sq[x] = a.sq[x];
  const int lc_raw = t / N3;
  const bool pad = lc_raw >= CPB;
  const int lc = pad ? CPB - 1 : lc_raw;
  const int pt = pad ? 0 : t - lc_raw * N3;
  Tile<N, Number> T;
  T.base = s_tile + lc * NTERM * N3;
  T.pt = pt;
  T.i = pt % N;
  T.j = (pt / N) % N;
  T.k = pt / (N * N);
  T.writer = !pad;
  const int first_cell = a.cell_begin + blockIdx.x * CPB, cell = first_cell + lc;
  const bool active = !pad && cell < a.cell_end;
  const int64_t qb = (int64_t)first_cell * N3;
  const uint32_t lo = active ? (uint32_t)t : 0u;
  const uint32_t entry = active ? (a.cell_nodes + qb)[lo] : 0u;
  uint32_t slot = 0;
  if constexpr (kToCells) slot = a.slots ? (a.slots + qb)[lo] : (uint32_t)(qb + lo);
  Number coef[NTERM];
  {
    typename QOp::Data qd = qop.load(qb, lo, CPB > 1 && !active ? 0 : pt);
    const typename QOp::Cell cd = qop.load_cell(active ? cell : first_cell);
    if constexpr (QOp::kNodalField) {
      __shared__ Number s_shape[N * N], s_colloc[N * N];
      if (t < N * N) {
        s_shape[t] = a.shape[t];
        s_colloc[t] = a.colloc[t];
      }
      const int64_t node = (int64_t)(entry & kNodeMaskDev);
      Number w[3], wg[3][3];
#pragma unroll
      for (int c = 0; c < 3; ++c) w[c] = active ? qop.u[node * 3 + c] : Number(0);
      evaluate_g<N, 3, Number>(T, s_shape, s_colloc, w, wg);
      qop.attach(qd, wg);
    }
    DiagonalTerms<QOp>::eval(qop, cd, qd, coef);
  }
  if (!active)
#pragma unroll
    for (int x = 0; x < NTERM; ++x) coef[x] = 0;
  const Number *SS = s_sq, *SD = s_sq + N * N, *DD = s_sq + 2 * N * N;
  __syncthreads();
#pragma unroll
  for (int x = 0; x < NTERM; ++x) T.put(x, coef[x]);
  __syncthreads();
  // z: m and zz share (SS, SS) afterwards
#pragma unroll
  for (int d = 0; d < NC; ++d) {
    Number *c = coef + 7 * d;
    c[0] = T.template line_t<2>(SS, T.k, 7 * d) + T.template line_t<2>(DD, T.k, 7 * d + 3);
    c[1] = T.template line_t<2>(SS, T.k, 7 * d + 1);
    c[2] = T.template line_t<2>(SS, T.k, 7 * d + 2);
    c[4] = T.template line_t<2>(SS, T.k, 7 * d + 4);
    c[5] = T.template line_t<2>(SD, T.k, 7 * d + 5);
    c[6] = T.template line_t<2>(SD, T.k, 7 * d + 6);
    // the component is done here: without it all components' lines are in
    // flight at once
    if constexpr (NC == 3)
      asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[4]), "+v"(c[5]), "+v"(c[6]) : : "memory");
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < NC; ++d)
#pragma unroll
    for (int x = 0; x < 7; ++x)
      if (x != 3) T.put(7 * d + x, coef[7 * d + x]);
  __syncthreads();
  // y: (m + zz), yy and yz share SS afterwards, xy and xz share SD
#pragma unroll
  for (int d = 0; d < NC; ++d) {
    Number *c = coef + 7 * d;
    c[0] = T.template line_t<1>(SS, T.j, 7 * d) + T.template line_t<1>(DD, T.j, 7 * d + 2) +
           T.template line_t<1>(SD, T.j, 7 * d + 6);
    c[1] = T.template line_t<1>(SS, T.j, 7 * d + 1);
    c[4] = T.template line_t<1>(SD, T.j, 7 * d + 4) + T.template line_t<1>(SS, T.j, 7 * d + 5);
    if constexpr (NC == 3) asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[4]) : : "memory");
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < NC; ++d) {
    T.put(7 * d, coef[7 * d]);
    T.put(7 * d + 1, coef[7 * d + 1]);
    T.put(7 * d + 4, coef[7 * d + 4]);
  }
  __syncthreads();
  if (!active) return;
  const int64_t node = entry & kNodeMaskDev;
  Number r[NC];
#pragma unroll
  for (int d = 0; d < NC; ++d)
    r[d] = T.template line_t<0>(SS, T.i, 7 * d) + T.template line_t<0>(DD, T.i, 7 * d + 1) +
           T.template line_t<0>(SD, T.i, 7 * d + 4);
  if constexpr (kToCells) {
    store_node<Number, NC>(a.diag + (int64_t)slot * NC, r);
  } else {
#pragma unroll
    for (int d = 0; d < NC; ++d)
      if (!((entry >> (kConstraintShift + d)) & 1u)) {
        Number *out = a.diag + node * NC + d;
        *out = (entry >> 31) ? r[d] : *out + r[d];
      }
  }
}

// GATHER: the nodes' sums in colour order, 1 on constrained components, and the
// inverse; flags entries that are not positive
template <typename Number, int NC>
__global__ void __launch_bounds__(kGatherThreads)
    diagonal_sums_kernel(GatherTables<Number> g, Number *__restrict__ diag, Number *__restrict__ inv, int64_t n_nodes,
                         int *flag) {
  const int64_t node = (int64_t)blockIdx.x * kGatherThreads + threadIdx.x;
  if (node >= n_nodes) return;
  const unsigned m = g.cmask[node];
  Number t[NC] = {}, r[NC];
  add_contributions<Number, NC>(g.contrib, g.index, g.offsets[node], g.offsets[node + 1], t);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if ((m >> c) & 1u) t[c] = Number(1);
    if (!(t[c] > Number(0))) *flag = 1;
    r[c] = Number(1) / t[c];
  }
  store_node<Number, NC>(diag + node * NC, t);
  store_node<Number, NC>(inv + node * NC, r);
}

}  // namespace mfg
