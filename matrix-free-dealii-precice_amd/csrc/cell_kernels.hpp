// Sum-factorisation cell kernels for gfx950 (CDNA4, wave64).
//
// Layout of one launch: a workgroup processes CPB cells, one thread per
// quadrature point (n_q = p+1, so points and nodes share the N^3 index space
// and the thread also owns node (i,j,k) of its cell).  The three 1D sweeps of
// each evaluate/integrate pass go through an LDS tile per cell; the
// collocation derivative at the Gauss points turns the three gradient
// directions into one LDS round trip.  Gather is a coalesced read of the
// int32 cell->node map followed by per-node vector loads.  Cells come in
// colours (no two cells of a colour share a node), one launch per colour, so
// the scatter is a plain read-modify-write, whose read is issued with the
// gather; the first colour that touches a node stores instead (bit 31 of its
// map entry), which makes vmult need no zero fill.  Constrained dofs are skipped via the constraint bits stored
// above bit 28 of every map entry.
//
// Algorithmic reference: FEEvaluation::evaluate/integrate with
// values|gradients as used by NeoHookOperator::do_operation_on_cell
// (mf_nh_operator.h:651-1019) and LaplaceOperator::do_operation_on_cell
// (heat_transfer.h:234-250).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "operator.hpp"
#include "smoother_terms.hpp"

namespace mfg {

constexpr int kConstraintShift = 28;
constexpr uint32_t kNodeMaskDev = (1u << kConstraintShift) - 1u;

template <int P, int CPB>
constexpr int block_threads() {
  return ((CPB * (P + 1) * (P + 1) * (P + 1) + 63) / 64) * 64;
}

// cells per workgroup of the apply / cache kernels, per degree.  Q4: one cell
// per workgroup measured 3-5 % faster than two for the solid and the heat
// operator in FP64 and, once the per-cell tables became scalar loads, 2-5 %
// in FP32.  Q3 and Q5 with one cell instead of two, Q2 with two cells (one
// wave) instead of seven, on 3-6M-DoF meshes: solid FP64 -4 to -30 %, heat
// -4 to -26 %, FP32 -1 to -3 %, small meshes unchanged.
template <int P, typename Number>
struct DefaultCPB {
  static constexpr int value = P == 1 ? 8 : P == 2 ? 2 : 1;
};

// Workgroups are dispatched round-robin over the 8 XCDs; remap so that each
// XCD walks one contiguous range of cells (shared nodes stay in one L2).
__device__ inline int xcd_remap(int b, int G) {
  const int x = b & 7, l = b >> 3, q = G >> 3, r = G & 7;
  return x * q + (x < r ? x : r) + l;
}


// Per-thread view of the cell tile in LDS.
template <int N, typename Number>
struct Tile {
  static constexpr int N3 = N * N * N;
  Number *base;  // slot 0 of this cell
  int i, j, k, pt;
  bool writer;   // false for padding lanes
  __device__ Number *slot(int s) const { return base + s * N3; }
  __device__ void put(int s, Number v) const {
    if (writer) base[s * N3 + pt] = v;
  }
  // sum_a M[row*N + a] * slot(a along dir)
  template <int DIR>
  __device__ Number line(const Number *M, int row, int s) const {
    const Number *src = slot(s);
    Number r = 0;
    if (DIR == 0) {
      const Number *b = src + N * (j + N * k);
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[row * N + a] * b[a];
    } else if (DIR == 1) {
      const Number *b = src + i + N * N * k;
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[row * N + a] * b[a * N];
    } else {
      const Number *b = src + i + N * j;
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[row * N + a] * b[a * N * N];
    }
    return r;
  }
  // sum_a M[a*N + col] * slot(a along dir)   (transposed matrix)
  template <int DIR>
  __device__ Number line_t(const Number *M, int col, int s) const {
    const Number *src = slot(s);
    Number r = 0;
    if (DIR == 0) {
      const Number *b = src + N * (j + N * k);
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[a * N + col] * b[a];
    } else if (DIR == 1) {
      const Number *b = src + i + N * N * k;
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[a * N + col] * b[a * N];
    } else {
      const Number *b = src + i + N * j;
#pragma unroll
      for (int a = 0; a < N; ++a) r += M[a * N + col] * b[a * N * N];
    }
    return r;
  }
};

// The gradient phase of evaluate_vg and the first phase of integrate_vg read
// 3 NC lines of N LDS values each.  Unrolled over the components, the
// compiler issues all of them at once; rolled, each line's reads wait for the
// one before, since the register-indexed result keeps them in order.  For
// N >= 6 the unrolled form's registers cost more than that (Q5 FP64 192 VGPRs
// against 124, 20M unknowns: 658 against 560 us).  For N = 5 the kernel with
// the 10-word point operation takes 106 VGPRs unrolled, 126 rolled: 487 -> 480
// us at 20M unknowns FP64, 39.7 -> 37.5 us at 0.2M (FP32 266 -> 264, 35.4 ->
// 33.1); the other point operations gain as well (formulation 0 649 -> 624,
// the folded words 544 -> 526; 3M unknowns: tensor4 209 -> 196, the folded words
// on non-affine cells 119 -> 110).  Two stay rolled: scalar_referential, which
// evaluates two fields (194 VGPRs unrolled), and the colour launches of
// tensor4_ns in FP64, whose 91 words per point keep the memory busy by
// themselves (3M unknowns 303 us unrolled, 272 rolled, 12M 1312 and 1195; its
// GATHER launch 22.3 and 25.1 at 0.2M, 102.5 and 98.0 at 1M).
template <int N, bool kRollN5 = false>
constexpr bool rolled_components() {
  return N >= (kRollN5 ? 5 : 6);
}

// Evaluate values and reference-coordinate gradients at the quadrature points
// of NC components; slots 0..2NC-1 are used.  On return the B slots hold the
// point values (still read by later lines until the next barrier).
template <int N, int NC, typename Number, bool kRolled = rolled_components<N>()>
__device__ inline void evaluate_vg(const Tile<N, Number> &T, const Number *S, const Number *D, const Number (&u)[NC],
                                   Number (&val)[NC], Number (&grad)[NC][3]) {
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(c, u[c]);
  __syncthreads();
  Number t[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) t[c] = T.template line<0>(S, T.i, c);
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(NC + c, t[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) t[c] = T.template line<1>(S, T.j, NC + c);
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(c, t[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) val[c] = T.template line<2>(S, T.k, c);
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(NC + c, val[c]);
  __syncthreads();
  auto gradient = [&](int c) {
    grad[c][0] = T.template line<0>(D, T.i, NC + c);
    grad[c][1] = T.template line<1>(D, T.j, NC + c);
    grad[c][2] = T.template line<2>(D, T.k, NC + c);
  };
  if constexpr (kRolled) {
#pragma unroll 1
    for (int c = 0; c < NC; ++c) gradient(c);
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) gradient(c);
  }
}

// Integrate submitted values and reference gradients back to the nodes
// (transpose of evaluate_vg).  Uses all 3NC slots; with kSpareSlots the tile
// has 5NC slots and the gradients go to slots 2NC.. that evaluate_vg does not
// use, which makes the two barriers that only guard slot reuse (after
// evaluate_vg's last reads and after the gradient lines) unnecessary.
template <int N, int NC, typename Number, bool kSpareSlots = false, bool kRolled = rolled_components<N>()>
__device__ inline void integrate_vg(const Tile<N, Number> &T, const Number *S, const Number *D,
                                    const Number (&val)[NC], const Number (&grad)[NC][3], Number (&out)[NC]) {
  constexpr int G0 = kSpareSlots ? 2 * NC : 0;  // first gradient slot
  if constexpr (!kSpareSlots) __syncthreads();  // B slots may still be read by evaluate_vg's last lines
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int f = 0; f < 3; ++f) T.put(G0 + 3 * c + f, grad[c][f]);
  __syncthreads();
  Number r[NC];
  auto gradient_t = [&](int c) {
    r[c] = val[c] + T.template line_t<0>(D, T.i, G0 + 3 * c + 0) + T.template line_t<1>(D, T.j, G0 + 3 * c + 1) +
           T.template line_t<2>(D, T.k, G0 + 3 * c + 2);
  };
  if constexpr (kRolled) {
#pragma unroll 1
    for (int c = 0; c < NC; ++c) gradient_t(c);
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) gradient_t(c);
  }
  if constexpr (!kSpareSlots) __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) r[c] = T.template line_t<2>(S, T.k, c);
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(NC + c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) r[c] = T.template line_t<1>(S, T.j, NC + c);
#pragma unroll
  for (int c = 0; c < NC; ++c) T.put(c, r[c]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) out[c] = T.template line_t<0>(S, T.i, c);
}

// Evaluate only reference gradients (cache()); same slot usage as evaluate_vg.
template <int N, int NC, typename Number, bool kRolled = rolled_components<N>()>
__device__ inline void evaluate_g(const Tile<N, Number> &T, const Number *S, const Number *D, const Number (&u)[NC],
                                  Number (&grad)[NC][3]) {
  Number val[NC];
  evaluate_vg<N, NC, Number, kRolled>(T, S, D, u, val, grad);
}

// The quadrature data is read once per operator application: load it
// non-temporally so that it does not evict from the caches the vector entries
// that the next colour reads again (nodes shared between cells).
template <typename Number>
__device__ inline Number stream_load(const Number *p) {
  return __builtin_nontemporal_load(p);
}

// Per-cell tables (geometry of affine cells) are read-only during a launch.
// Read through the constant address space: where the cell index is uniform
// across the wave (one cell per workgroup) the loads become scalar loads into
// SGPRs, otherwise they stay vector loads.
template <typename Number>
using ConstantPtr = const Number __attribute__((address_space(4))) *;
template <typename Number>
__device__ inline ConstantPtr<Number> as_constant(const Number *p) {
  return (ConstantPtr<Number>)p;
}

// ------------------------------------------------------ quadrature ops ---
// Each op provides
//   load_cell(cell) -> Cell          what is constant on a stored cell,
//   load(qb, lo, pt) -> Data         the fields of point qb + lo = cell N^3 + pt
//                                    (qb the same on every lane: the loads take
//                                    a scalar base and a 32-bit lane offset),
//   apply_grad(Cell, Data, grad)     reference gradients at the point -> the
//                                    submitted reference gradients, with JxW,
//   value_scale(Cell, Data)          the factor of the submitted values
// (apply: both).
struct NoCell {};
template <class QOp, typename Number, int NC>
__device__ inline void apply_qop(const QOp &qop, const typename QOp::Cell &cd, const typename QOp::Data &d,
                                 Number (&val)[NC], Number (&grad)[NC][3]) {
  qop.apply_grad(cd, d, grad);
  const Number s = qop.value_scale(cd, d);
#pragma unroll
  for (int c = 0; c < NC; ++c) val[c] = s * val[c];
}

// symmetric index pairs xx, yy, zz, xy, xz, yz
constexpr int kSymI[6] = {0, 1, 2, 0, 0, 1}, kSymJ[6] = {0, 1, 2, 1, 2, 2};

// Solid, tensor2 caching, formulation 1 (mf_nh_operator.h:945-974).
// The reference caches, per point, the current-frame Jinv and JxW (from
// MappingQEulerian) and the scalars 2 s / J, 1 / J and tau / J, where
// s = mu - 2 lambda ln J and tau is the Kirchhoff stress.  The operator only
// uses them multiplied by the current JxW = JxW_ref J, so these products are
// cached instead:
//   fields 0..8   Jinv_cur[f][e]
//   field  9      JxW_ref s
//   fields 10..15 JxW_ref tau (xx, yy, zz, xy, xz, yz)
//   field  16     JxW_ref, only on meshes with a cell that is not affine in the
//                 reference configuration.  Otherwise JxW_ref = w_q det J_ref
//                 comes from one word per cell (cell_jxw) and the tensor
//                 weights (wq).
// 16 words per point instead of the reference's 18, and no JxW products in
// the point operation.
// kStreamLast: field 16 is loaded past the caches.  It stays in the 256 MB MALL
// from one application to the next where it is a good part smaller; above, it
// only drives the vectors out.  Non-affine Q1 FP64, streamed / cached: 5M
// unknowns (a field of 107 MB) 432 / 414 us, 10M (213 MB) 824 / 836, 15M 1269 /
// 1373; Q4 2M (10 MB) 97 / 89.  A type of its own: with cell_jxw decided at run
// time the compiler merges the two loads into a plain one.
template <typename Number, bool kStreamLast = false>
struct QSolidT2F1 {
  static constexpr int NC = 3;
  static constexpr int kFields = 17;  // 16 with cell_jxw
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number two_lambda, rho_alpha;
  const Number *cell_jxw;  // det J_ref per stored cell, or null: field 16 holds JxW_ref
  const Number *wq;        // N^3 tensor-product quadrature weights (with cell_jxw)
  struct Cell {
    Number jxw;
  };
  struct Data {
    Number ji[9], s, T[6], w;  // w: the point's quadrature weight (with cell_jxw) or JxW_ref
  };
  __device__ Cell load_cell(int cell) const {
    return Cell{!kStreamLast && cell_jxw ? as_constant(cell_jxw)[cell] : Number(1)};
  }
  __device__ Number jxw(const Cell &cd, const Data &d) const { return cd.jxw * d.w; }
  // fields 0..15 are stored in pairs, qd[((f / 2) nqp + q) 2 + f % 2], field
  // 16 plainly after them: 8 16-byte (FP64) loads bring a point's 16 words
  typedef Number Pair __attribute__((ext_vector_type(2)));
  __device__ Data load(int64_t qb, uint32_t lo, int pt) const {
    Data d;
    Number f16[16];
    const Pair *qp = reinterpret_cast<const Pair *>(qd);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const Pair x = __builtin_nontemporal_load(qp + k * nqp + qb + lo);
      f16[2 * k] = x.x;
      f16[2 * k + 1] = x.y;
    }
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ji[f] = f16[f];
    d.s = f16[9];
#pragma unroll
    for (int f = 0; f < 6; ++f) d.T[f] = f16[10 + f];
    if constexpr (kStreamLast) d.w = stream_load(qd + 16 * nqp + qb + lo);
    else d.w = cell_jxw ? wq[pt] : qd[16 * nqp + qb + lo];
    return d;
  }
  __device__ Number value_scale(const Cell &cd, const Data &d) const { return rho_alpha * jxw(cd, d); }
  __device__ void apply_grad(const Cell &cd, const Data &d, Number (&grad)[3][3]) const {
    const Number w = jxw(cd, d);
    Number g[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) g[c][e] = grad[c][0] * d.ji[0 * 3 + e] + grad[c][1] * d.ji[1 * 3 + e] + grad[c][2] * d.ji[2 * 3 + e];
    const Number tr = g[0][0] + g[1][1] + g[2][2];
    const Number diag = two_lambda * w * tr;
    // T symmetric: T[0]=xx T[1]=yy T[2]=zz T[3]=xy T[4]=xz T[5]=yz
    const Number Tm[3][3] = {{d.T[0], d.T[3], d.T[4]}, {d.T[3], d.T[1], d.T[5]}, {d.T[4], d.T[5], d.T[2]}};
    Number Pm[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b)
        Pm[a][b] = d.s * (g[a][b] + g[b][a]) + (a == b ? diag : Number(0)) + g[a][0] * Tm[0][b] +
                   g[a][1] * Tm[1][b] + g[a][2] * Tm[2][b];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int f = 0; f < 3; ++f)
        grad[c][f] = Pm[c][0] * d.ji[f * 3 + 0] + Pm[c][1] * d.ji[f * 3 + 1] + Pm[c][2] * d.ji[f * 3 + 2];
  }
};

// Solid, tensor2 caching, formulation 1, from 10 words per point on affine
// meshes: the operator of QSolidT2F1 with the stress products pulled back to
// the reference cell.  With g = Grad_xi v Jinv_cur the spatial gradient,
// s = mu - 2 lambda ln J and tau = mu F F^T - s I,
//   s (g + g^T) + 2 lambda tr(g) I + g tau = s g^T + 2 lambda tr(g) I + mu g F F^T,
// and with Jinv_cur = J_ref^{-1} F^{-1} the last term, multiplied by
// Jinv_cur^T, is mu Grad_xi v (J_ref^{-1} J_ref^{-T}): it needs neither F nor
// tau, only the metric G = J_ref^{-1} J_ref^{-T}, constant per cell.  With
// M = Jinv_cur Grad_xi v the submitted gradient is
//   w [ mu Grad_xi v G + ((s M + 2 lambda tr(M) I) Jinv_cur)^T ],
// w = JxW_ref = det J_ref w_q.  Fields: Jinv_cur[f][e] (9), s; stored in pairs
// of fields (below).
// kEarlyCell (the cell index is the same on every lane: one cell per
// workgroup): the cell's G and det J_ref are loaded into SGPRs with the point
// data, so that their latency overlaps the gather's instead of following the
// evaluate sweeps.
// kCartesian (every cell's J_ref is diagonal, as on axis-aligned boxes): only
// the 3 diagonal entries of G are loaded, and the products with the exact
// zeros off the diagonal are left out.  Every rounding step of the general
// form survives, so the two agree bit for bit (up to the sign of a zero).
// Measured against rebuilding Jinv_cur, F and tau per point from Grad_xi u
// (about 90 instead of 200 FP64 operations per point and no division; the
// same 10 words): Q4 beam of 128x32x32 cells FP64 0.647 -> 0.605 ms per vmult
// (2.76 -> 2.95 TB/s of the data held), 96x24x24 cells FP32 0.167 -> 0.161 ms,
// Q2 37x29x23 cells FP64 44.5 -> 41.3 us.
template <typename Number, bool kEarlyCell = false, bool kCartesian = false>
struct QSolidT2F1G {
  static constexpr int NC = 3;
  static constexpr int kFields = 10;
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number mu, two_lambda, rho_alpha;
  const Number *cell_met;  // per stored cell: G (xx, yy, zz, xy, xz, yz)
  const Number *cell_jxw;  // det J_ref per stored cell
  const Number *wq;        // N^3 tensor-product quadrature weights
  struct Cell {
    Number jxw, g[kCartesian ? 3 : 6];  // det J_ref; G or its diagonal
  };
  struct Data {
    Number ji[9], s, w;  // w: the point's quadrature weight
  };
  __device__ Cell load_cell(int cell) const {
    Cell cd;
    const ConstantPtr<Number> m = as_constant(cell_met) + (int64_t)cell * 6;
    cd.jxw = as_constant(cell_jxw)[cell];
#pragma unroll
    for (int f = 0; f < (kCartesian ? 3 : 6); ++f) cd.g[f] = m[f];
    if constexpr (kEarlyCell) {
      // all values in SGPRs here: one wait, before the first barrier
      if constexpr (kCartesian)
        asm volatile("" : "+s"(cd.jxw), "+s"(cd.g[0]), "+s"(cd.g[1]), "+s"(cd.g[2]));
      else
        asm volatile(""
                     : "+s"(cd.jxw), "+s"(cd.g[0]), "+s"(cd.g[1]), "+s"(cd.g[2]), "+s"(cd.g[3]), "+s"(cd.g[4]),
                       "+s"(cd.g[5]));
    }
    return cd;
  }
  // fields are stored in pairs, qd[((f / 2) nqp + q) 2 + f % 2]: one 16-byte
  // (FP64) load brings two fields of a point
  typedef Number Pair __attribute__((ext_vector_type(2)));
  __device__ Data load(int64_t qb, uint32_t lo, int pt) const {
    Data d;
    const Pair *qp = reinterpret_cast<const Pair *>(qd);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const Pair x = __builtin_nontemporal_load(qp + k * nqp + qb + lo);
      d.ji[2 * k] = x.x;
      if (k < 4) d.ji[2 * k + 1] = x.y;
      else d.s = x.y;
    }
    d.w = wq[pt];
    return d;
  }
  __device__ Number value_scale(const Cell &cd, const Data &d) const { return rho_alpha * (cd.jxw * d.w); }
  __device__ void apply_grad(const Cell &cd, const Data &d, Number (&grad)[3][3]) const {
    const Number w = cd.jxw * d.w;
    const Number *ji = d.ji;
    Number M[3][3];
#pragma unroll
    for (int f = 0; f < 3; ++f)
#pragma unroll
      for (int h = 0; h < 3; ++h) M[f][h] = ji[f * 3 + 0] * grad[0][h] + ji[f * 3 + 1] * grad[1][h] + ji[f * 3 + 2] * grad[2][h];
    const Number sw = w * d.s, wm = w * mu;
    const Number diag = two_lambda * w * (M[0][0] + M[1][1] + M[2][2]);
#pragma unroll
    for (int f = 0; f < 3; ++f)
#pragma unroll
      for (int h = 0; h < 3; ++h) M[f][h] = f == h ? sw * M[f][h] + diag : sw * M[f][h];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      Number t[3];  // row c of Grad_xi v G
      if constexpr (kCartesian) {
        // the general form's sum of three products, two of them exact zeros,
        // rounds as this one product does
#pragma unroll
        for (int f = 0; f < 3; ++f) t[f] = grad[c][f] * cd.g[f];
      } else {
        t[0] = grad[c][0] * cd.g[0] + grad[c][1] * cd.g[3] + grad[c][2] * cd.g[4];
        t[1] = grad[c][0] * cd.g[3] + grad[c][1] * cd.g[1] + grad[c][2] * cd.g[5];
        t[2] = grad[c][0] * cd.g[4] + grad[c][1] * cd.g[5] + grad[c][2] * cd.g[2];
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        const Number r = M[f][0] * ji[0 * 3 + c] + M[f][1] * ji[1 * 3 + c] + M[f][2] * ji[2 * 3 + c];
        grad[c][f] = wm * t[f] + r;
      }
    }
  }
};

// Solid, tensor2 caching, formulation 0 (mf_nh_operator.h:701-840).
// Fields: Jinv_cur (9), JxW, J^{-1/3}, F (9).
template <typename Number>
struct QSolidT2F0 {
  static constexpr int NC = 3;
  static constexpr int kFields = 20;
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number kappa, c_1, rho_alpha;
  using Cell = NoCell;
  __device__ Cell load_cell(int) const { return Cell{}; }
  struct Data {
    Number ji[9], jxw, jm13, F[9];
  };
  __device__ Data load(int64_t qb, uint32_t lo, int) const {
    Data d;
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ji[f] = stream_load(qd + f * nqp + qb + lo);
    d.jxw = stream_load(qd + 9 * nqp + qb + lo);
    d.jm13 = stream_load(qd + 10 * nqp + qb + lo);
#pragma unroll
    for (int f = 0; f < 9; ++f) d.F[f] = stream_load(qd + (11 + f) * nqp + qb + lo);
    return d;
  }
  __device__ static Number det(const Number *F) {
    return F[0] * (F[4] * F[8] - F[5] * F[7]) - F[1] * (F[3] * F[8] - F[5] * F[6]) + F[2] * (F[3] * F[7] - F[4] * F[6]);
  }
  __device__ Number value_scale(const Cell &, const Data &d) const {
    const Number inv_det = Number(1) / det(d.F);
    return d.jxw * rho_alpha * inv_det;
  }
  __device__ void apply_grad(const Cell &, const Data &d, Number (&grad)[3][3]) const {
    Number g[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) g[c][e] = grad[c][0] * d.ji[0 * 3 + e] + grad[c][1] * d.ji[1 * 3 + e] + grad[c][2] * d.ji[2 * 3 + e];
    const Number *F = d.F;
    const Number det_F = det(F);
    Number Fb[9];
#pragma unroll
    for (int a = 0; a < 9; ++a) Fb[a] = F[a] * d.jm13;
    Number tau_bar[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b)
        tau_bar[a][b] = Number(2) * c_1 * (Fb[a * 3 + 0] * Fb[b * 3 + 0] + Fb[a * 3 + 1] * Fb[b * 3 + 1] + Fb[a * 3 + 2] * Fb[b * 3 + 2]);
    const Number tr_tau_bar = tau_bar[0][0] + tau_bar[1][1] + tau_bar[2][2];
    const Number tr_tau_bar_dim = tr_tau_bar / Number(3);
    const Number inv_det = Number(1) / det_F;
    const Number dPsi = (kappa / Number(2)) * (det_F - inv_det);
    const Number dPsi_J = dPsi * det_F;
    const Number d2Psi = (kappa / Number(2)) * (Number(1) + inv_det * inv_det);
    Number s[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) s[a][b] = Number(0.5) * (g[a][b] + g[b][a]);
    const Number tr = s[0][0] + s[1][1] + s[2][2];
    Number tau_iso_src = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) tau_iso_src += (tau_bar[a][b] - (a == b ? tr_tau_bar_dim : Number(0))) * s[a][b];
    const Number vol = det_F * (dPsi + det_F * d2Psi) * tr;
    Number Pm[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const Number tau_iso = tau_bar[a][b] - (a == b ? tr_tau_bar_dim : Number(0));
        const Number dev = s[a][b] - (a == b ? tr / Number(3) : Number(0));
        Number jc = s[a][b] * (-dPsi_J * Number(2)) + Number(2.0 / 3.0) * tr_tau_bar * dev -
                    Number(2.0 / 3.0) * tr * tau_iso;
        if (a == b) jc += vol - Number(2.0 / 3.0) * tau_iso_src;
        Number geo = 0;
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const Number tau_mb = tau_bar[m][b] + (m == b ? dPsi_J - tr_tau_bar_dim : Number(0));
          geo += g[a][m] * tau_mb;
        }
        Pm[a][b] = (jc + geo) * inv_det;
      }
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int f = 0; f < 3; ++f)
        grad[c][f] = d.jxw * (Pm[c][0] * d.ji[f * 3 + 0] + Pm[c][1] * d.ji[f * 3 + 1] + Pm[c][2] * d.ji[f * 3 + 2]);
  }
};

// Heat: value v, gradient c*dt*grad v (heat_transfer.h:242-248).  On the
// reference cell the gradient term is c dt JxW G Grad_xi v with the metric
// G = Jinv Jinv^T (symmetric).  Fields: Jinv (9), JxW, c per point; or, when
// every cell is affine (the affine-cell geometry of MatrixFree), G and det J
// once per cell (cell_geo, 7 words), JxW = det J * wq[point], and c the only
// field.
template <typename Number, bool kAffine>
struct QHeat {
  static constexpr int NC = 1;
  static constexpr int kFields = kAffine ? 1 : 11;
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number dt;
  const Number *cell_geo;  // kAffine, per stored cell: G (xx, yy, zz, xy, xz, yz), det J
  const Number *wq;        // N^3 tensor-product quadrature weights (kAffine)
  struct Cell {
    Number g[6], det;
  };
  struct Data {
    Number ji[kAffine ? 1 : 9], w, c;  // w: the point's quadrature weight (kAffine) or JxW
  };
  __device__ Cell load_cell(int cell) const {
    Cell cd{};
    if constexpr (kAffine) {
      const ConstantPtr<Number> g = as_constant(cell_geo) + (int64_t)cell * 7;
#pragma unroll
      for (int f = 0; f < 6; ++f) cd.g[f] = g[f];
      cd.det = g[6];
    }
    return cd;
  }
  __device__ Data load(int64_t qb, uint32_t lo, int pt) const {
    Data d;
    if constexpr (kAffine) {
      d.w = wq[pt];
      d.c = stream_load(qd + qb + lo);
    } else {
#pragma unroll
      for (int f = 0; f < 9; ++f) d.ji[f] = stream_load(qd + f * nqp + qb + lo);
      d.w = stream_load(qd + 9 * nqp + qb + lo);
      d.c = stream_load(qd + 10 * nqp + qb + lo);
    }
    return d;
  }
  __device__ Number value_scale(const Cell &cd, const Data &d) const { return kAffine ? cd.det * d.w : d.w; }
  __device__ void apply_grad(const Cell &cd, const Data &d, Number (&grad)[1][3]) const {
    const Number s = d.c * dt * value_scale(cd, d);
    const Number g0 = grad[0][0], g1 = grad[0][1], g2 = grad[0][2];
    if constexpr (kAffine) {
      grad[0][0] = s * (cd.g[0] * g0 + cd.g[3] * g1 + cd.g[4] * g2);
      grad[0][1] = s * (cd.g[3] * g0 + cd.g[1] * g1 + cd.g[5] * g2);
      grad[0][2] = s * (cd.g[4] * g0 + cd.g[5] * g1 + cd.g[2] * g2);
    } else {
      Number gx[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) gx[e] = g0 * d.ji[e] + g1 * d.ji[3 + e] + g2 * d.ji[6 + e];
#pragma unroll
      for (int f = 0; f < 3; ++f)
        grad[0][f] = s * (gx[0] * d.ji[f * 3] + gx[1] * d.ji[f * 3 + 1] + gx[2] * d.ji[f * 3 + 2]);
    }
  }
};

// The other formulation-1 cachings (MF caching parameter,
// mf_nh_operator.h:848-1010).  They define the same operator as tensor2 and
// trade memory for arithmetic differently.

// scalar_referential (mf_nh_operator.h:848-943): reference-frame geometry
// and one scalar per point; F is rebuilt from the cached nodal displacement
// at every application.  Fields: Jinv_ref (9), JxW_ref, mu - 2 lambda ln J.
template <typename Number>
struct QSolidSR {
  static constexpr int NC = 3;
  static constexpr int kFields = 11;
  static constexpr bool kNodalField = true;  // reference gradient of u at the point, set by attach()
  const Number *qd;
  int64_t nqp;
  const Number *u;  // nodal linearisation point, 3 per node
  Number mu, two_lambda, rho_alpha;
  using Cell = NoCell;
  __device__ Cell load_cell(int) const { return Cell{}; }
  struct Data {
    Number ji[9], jxw, sc, ug[9];
  };
  __device__ Data load(int64_t qb, uint32_t lo, int) const {
    Data d;
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ji[f] = stream_load(qd + f * nqp + qb + lo);
    d.jxw = stream_load(qd + 9 * nqp + qb + lo);
    d.sc = stream_load(qd + 10 * nqp + qb + lo);
    return d;
  }
  __device__ void attach(Data &d, const Number (&ug)[3][3]) const {
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ug[f] = ug[f / 3][f % 3];
  }
  __device__ Number value_scale(const Cell &, const Data &d) const { return d.jxw * rho_alpha; }
  __device__ void apply_grad(const Cell &, const Data &d, Number (&grad)[3][3]) const {
    Number g[3][3], F[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        g[c][e] = grad[c][0] * d.ji[0 * 3 + e] + grad[c][1] * d.ji[1 * 3 + e] + grad[c][2] * d.ji[2 * 3 + e];
        F[c][e] = d.ug[c * 3 + 0] * d.ji[0 * 3 + e] + d.ug[c * 3 + 1] * d.ji[1 * 3 + e] +
                  d.ug[c * 3 + 2] * d.ji[2 * 3 + e] + (c == e ? Number(1) : Number(0));
      }
    const Number det = F[0][0] * (F[1][1] * F[2][2] - F[1][2] * F[2][1]) - F[0][1] * (F[1][0] * F[2][2] - F[1][2] * F[2][0]) +
                       F[0][2] * (F[1][0] * F[2][1] - F[1][1] * F[2][0]);
    const Number id = Number(1) / det;
    Number Fi[3][3];
    Fi[0][0] = (F[1][1] * F[2][2] - F[1][2] * F[2][1]) * id;
    Fi[0][1] = (F[0][2] * F[2][1] - F[0][1] * F[2][2]) * id;
    Fi[0][2] = (F[0][1] * F[1][2] - F[0][2] * F[1][1]) * id;
    Fi[1][0] = (F[1][2] * F[2][0] - F[1][0] * F[2][2]) * id;
    Fi[1][1] = (F[0][0] * F[2][2] - F[0][2] * F[2][0]) * id;
    Fi[1][2] = (F[0][2] * F[1][0] - F[0][0] * F[1][2]) * id;
    Fi[2][0] = (F[1][0] * F[2][1] - F[1][1] * F[2][0]) * id;
    Fi[2][1] = (F[0][1] * F[2][0] - F[0][0] * F[2][1]) * id;
    Fi[2][2] = (F[0][0] * F[1][1] - F[0][1] * F[1][0]) * id;
    // the stress products on the reference configuration (as in
    // QSolidT2F1G): mu Grad v + ((s A + 2 lambda tr(A) I) F^{-1})^T with
    // A = F^{-1} Grad v, then to reference-cell gradients
    Number A[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) A[a][b] = Fi[a][0] * g[0][b] + Fi[a][1] * g[1][b] + Fi[a][2] * g[2][b];
    const Number diag = two_lambda * (A[0][0] + A[1][1] + A[2][2]);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) A[a][b] = a == b ? d.sc * A[a][b] + diag : d.sc * A[a][b];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      Number Pm[3];
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const Number r = A[b][0] * Fi[0][c] + A[b][1] * Fi[1][c] + A[b][2] * Fi[2][c];
        Pm[b] = mu * g[c][b] + r;
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) grad[c][f] = d.jxw * (Pm[0] * d.ji[f * 3 + 0] + Pm[1] * d.ji[f * 3 + 1] + Pm[2] * d.ji[f * 3 + 2]);
    }
  }
};

// tensor4 (mf_nh_operator.h:976-994): deformed-frame geometry, 1/J, tau/J
// and the symmetric fourth-order tangent C = (2 s_c/J) S + (2 lambda/J) I x I
// as a 6 x 6 table over the symmetric index pairs (xx,yy,zz,xy,xz,yz).
// Fields: Jinv_cur (9), JxW_cur, 1/J, tau/J (6), C (36); the C entries are
// read while contracting.
template <typename Number>
struct QSolidT4 {
  static constexpr int NC = 3;
  static constexpr int kFields = 53;
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number rho_alpha;
  using Cell = NoCell;
  __device__ Cell load_cell(int) const { return Cell{}; }
  struct Data {
    Number ji[9], jxw, c1, T[6];
    int64_t q;
  };
  __device__ Data load(int64_t qb, uint32_t lo, int) const {
    Data d;
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ji[f] = stream_load(qd + f * nqp + qb + lo);
    d.jxw = stream_load(qd + 9 * nqp + qb + lo);
    d.c1 = stream_load(qd + 10 * nqp + qb + lo);
#pragma unroll
    for (int f = 0; f < 6; ++f) d.T[f] = stream_load(qd + (11 + f) * nqp + qb + lo);
    d.q = qb + lo;
    return d;
  }
  __device__ Number value_scale(const Cell &, const Data &d) const { return d.jxw * rho_alpha * d.c1; }
  __device__ void apply_grad(const Cell &, const Data &d, Number (&grad)[3][3]) const {
    Number g[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) g[c][e] = grad[c][0] * d.ji[0 * 3 + e] + grad[c][1] * d.ji[1 * 3 + e] + grad[c][2] * d.ji[2 * 3 + e];
    // C : sym(g), summing both orders of the off-diagonal pairs
    Number sym2[6];
#pragma unroll
    for (int t = 0; t < 6; ++t)
      sym2[t] = (t < 3 ? Number(0.5) : Number(1)) * (g[kSymI[t]][kSymJ[t]] + g[kSymJ[t]][kSymI[t]]);
    Number Cs[6];
#pragma unroll
    for (int s6 = 0; s6 < 6; ++s6) {
      Number acc = 0;
#pragma unroll
      for (int t = 0; t < 6; ++t) acc += stream_load(qd + (17 + 6 * s6 + t) * nqp + d.q) * sym2[t];
      Cs[s6] = acc;
    }
    const Number Cm[3][3] = {{Cs[0], Cs[3], Cs[4]}, {Cs[3], Cs[1], Cs[5]}, {Cs[4], Cs[5], Cs[2]}};
    const Number Tm[3][3] = {{d.T[0], d.T[3], d.T[4]}, {d.T[3], d.T[1], d.T[5]}, {d.T[4], d.T[5], d.T[2]}};
    Number Pm[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) Pm[a][b] = Cm[a][b] + g[a][0] * Tm[0][b] + g[a][1] * Tm[1][b] + g[a][2] * Tm[2][b];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int f = 0; f < 3; ++f)
        grad[c][f] = d.jxw * (Pm[c][0] * d.ji[f * 3 + 0] + Pm[c][1] * d.ji[f * 3 + 1] + Pm[c][2] * d.ji[f * 3 + 2]);
    }
  }
};

// tensor4_ns (mf_nh_operator.h:996-1010): reference-frame geometry and the
// full (non-symmetric) fourth-order tangent A (81 entries), contracted as
// double_contract<2,0,3,1>(A, Grad v).  Fields: Jinv_ref (9), JxW_ref, A (81).
template <typename Number>
struct QSolidT4NS {
  static constexpr int NC = 3;
  static constexpr int kFields = 91;
  static constexpr bool kNodalField = false;
  const Number *qd;
  int64_t nqp;
  Number rho_alpha;
  using Cell = NoCell;
  __device__ Cell load_cell(int) const { return Cell{}; }
  struct Data {
    Number ji[9], jxw;
    int64_t q;
  };
  __device__ Data load(int64_t qb, uint32_t lo, int) const {
    Data d;
#pragma unroll
    for (int f = 0; f < 9; ++f) d.ji[f] = stream_load(qd + f * nqp + qb + lo);
    d.jxw = stream_load(qd + 9 * nqp + qb + lo);
    d.q = qb + lo;
    return d;
  }
  __device__ Number value_scale(const Cell &, const Data &d) const { return d.jxw * rho_alpha; }
  __device__ void apply_grad(const Cell &, const Data &d, Number (&grad)[3][3]) const {
    Number g[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 3; ++e) g[c][e] = grad[c][0] * d.ji[0 * 3 + e] + grad[c][1] * d.ji[1 * 3 + e] + grad[c][2] * d.ji[2 * 3 + e];
    Number Pm[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        Number acc = 0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int l = 0; l < 3; ++l) acc += stream_load(qd + (10 + ((a * 3 + b) * 3 + k) * 3 + l) * nqp + d.q) * g[k][l];
        Pm[a][b] = acc;
      }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int f = 0; f < 3; ++f)
        grad[c][f] = d.jxw * (Pm[c][0] * d.ji[f * 3 + 0] + Pm[c][1] * d.ji[f * 3 + 1] + Pm[c][2] * d.ji[f * 3 + 2]);
    }
  }
};

// ------------------------------------------------------ apply kernel ---
// One launch covers the cells [cell_begin, cell_end) of one colour: no two of
// them share a node, so the scatter is a plain read-modify-write and the
// result is bit-reproducible (cells are stored colour-major).
// fix_mode: 0 no constrained-row handling, 1 dst[c] = src[c], 2 dst[c] += src[c]
template <typename Number>
struct ApplyArgs {
  const uint32_t *cell_nodes;
  int cell_begin, cell_end;
  const Number *src;
  Number *dst;
  const Number *shape;   // N x N
  const Number *colloc;  // N x N
  const int32_t *constrained;
  int64_t n_constrained;
  int fix_mode;
  const uint32_t *slots;  // GATHER: where each (stored cell, point) puts its contribution; null: in point order
};

// The cells [cell_begin, min(cell_begin + cpb, cell_end)) on all threads of
// the workgroup, thread t owning point t % N3 of local cell t / N3; threads
// past cpb*N3 only join the barriers.  `assign`: the first colour touching a
// node stores instead of adding.  Shape and collocation tables must be in LDS
// before the first barrier inside.  kToCells: instead of the read-modify-write
// of dst, each point stores its node's contribution (NC values) at
// dst[slot NC + c], slot = slots[cell N3 + point] or (slots null) the point's
// number, for the gather of the GATHER schedule.
// The NC values of one node, loaded as one struct so that the compiler can use
// wide loads (nodes are 8-byte aligned; the hardware takes unaligned wide loads).
template <typename Number, int NC>
struct NodeValues {
  Number v[NC];
};
template <typename Number, int NC>
__device__ inline NodeValues<Number, NC> load_node(const Number *p) {
  return *reinterpret_cast<const NodeValues<Number, NC> *>(p);
}
template <typename Number, int NC>
__device__ inline void store_node(Number *p, const Number (&v)[NC]) {
  NodeValues<Number, NC> x;
#pragma unroll
  for (int c = 0; c < NC; ++c) x.v[c] = v[c];
  *reinterpret_cast<NodeValues<Number, NC> *>(p) = x;
}

// g_shape / g_colloc: the N x N 1D matrices in global memory, copied into
// s_shape / s_colloc here.  The LDS tile and the two tables must not be in use
// by other threads of the workgroup on entry (a caller that runs several
// groups in sequence puts a barrier between them).
template <int P, typename Number, class QOp, bool kToCells = false, bool kSpareSlots = false>
__device__ inline void cell_group(const QOp &qop, const uint32_t *__restrict__ cell_nodes,
                                  const Number *__restrict__ src, Number *__restrict__ dst, int cell_begin,
                                  int cell_end, int cpb, int assign, const Number *__restrict__ g_shape,
                                  const Number *__restrict__ g_colloc, Number *s_shape, Number *s_colloc,
                                  Number *s_tile, const uint32_t *__restrict__ slots = nullptr) {
  constexpr int N = P + 1, N3 = N * N * N, NC = QOp::NC;
  constexpr bool kRollN5 = QOp::kNodalField || (!kToCells && std::is_same<QOp, QSolidT4NS<double>>::value);
  constexpr bool kRolled = rolled_components<N, kRollN5>();
  const int t = threadIdx.x;
  const int lc_raw = t / N3;
  const bool pad = lc_raw >= cpb;
  const int lc = pad ? cpb - 1 : lc_raw;
  const int pt = pad ? 0 : t - lc_raw * N3;
  Tile<N, Number> T;
  T.base = s_tile + lc * (kSpareSlots ? 5 : 3) * NC * N3;
  T.pt = pt;
  T.i = pt % N;
  T.j = (pt / N) % N;
  T.k = pt / (N * N);
  T.writer = !pad;
  const int cell = cell_begin + lc;
  const bool active = !pad && cell < cell_end;
  // this thread's point: a base that is the same on every lane and a 32-bit
  // lane offset (threads without a point stay on the group's first)
  const int64_t qb = (int64_t)__builtin_amdgcn_readfirstlane(cell_begin) * N3;
  const uint32_t lo = active ? (uint32_t)t : 0u;

  uint32_t entry = active ? (cell_nodes + qb)[lo] : 0u;
  uint32_t slot = 0;
  if constexpr (kToCells) slot = slots ? (slots + qb)[lo] : (uint32_t)(qb + lo);
  // the 1D matrices are loaded with the map and written to LDS just before
  // the first barrier of the sweeps, which publishes them: no wait on these
  // loads stands before the gather
  const bool table_lane = t < N * N;
  Number sh = 0, co = 0;
  if (table_lane) {
    sh = g_shape[t];
    co = g_colloc[t];
  }
  const int64_t node = entry & kNodeMaskDev;
  // a node's NC values are contiguous: one wide load (FP64, NC = 3: a 16- and
  // an 8-byte load instead of three) for all components, constrained ones
  // dropped afterwards
  Number u[NC];
  {
    const NodeValues<Number, NC> v = active ? load_node<Number, NC>(src + node * NC) : NodeValues<Number, NC>{};
#pragma unroll
    for (int c = 0; c < NC; ++c) u[c] = ((entry >> (kConstraintShift + c)) & 1u) ? Number(0) : v.v[c];
  }
  // dst of this node: no other workgroup of the launch writes it, so the
  // scatter at the end is a plain store.  The first colour touching a node
  // stores without reading.  Read with the gather, the load's latency hides
  // behind the sweeps; read after them, its 2 NC registers are free during
  // the sweeps.  For the FP64 solid ops with per-point tensors and p <= 4 the
  // late read gives the kernel one more wave per SIMD and is the faster of the
  // two (measured); for the heat op and the 10-word tensor2 op, whose wave
  // count it does not change, and elsewhere the early read is.
  constexpr bool kLateDst = sizeof(Number) == 8 && P <= 4 && NC == 3 &&
                            !std::is_same<QOp, QSolidT2F1G<Number>>::value &&
                            !std::is_same<QOp, QSolidT2F1G<Number, true>>::value &&
                            !std::is_same<QOp, QSolidT2F1G<Number, true, true>>::value;
  const bool first = assign && (entry >> 31);
  Number dold[NC];
  if constexpr (!kLateDst && !kToCells) {
    // constrained components are read but not used: their dst entries are not stored
    const NodeValues<Number, NC> v =
        active && !first ? load_node<Number, NC>(dst + node * NC) : NodeValues<Number, NC>{};
#pragma unroll
    for (int c = 0; c < NC; ++c) dold[c] = v.v[c];
  }
  // the cached nodal field of the nodal-field ops, gathered with src
  NodeValues<Number, 3> w{};
  if constexpr (QOp::kNodalField) {
    if (active) w = load_node<Number, 3>(qop.u + node * 3);
  }
  // one cell per workgroup: the cell index is the same on every lane (padding
  // lanes included), which lets the per-cell tables come in as scalar loads
  const int qcell = cpb == 1 ? __builtin_amdgcn_readfirstlane(cell < cell_end ? cell : 0) : (active ? cell : 0);
  typename QOp::Data qd = qop.load(qb, lo, pt);
  const typename QOp::Cell cd = qop.load_cell(qcell);
  // read only after the barrier that follows the first puts of the sweeps
  if (table_lane) {
    s_shape[t] = sh;
    s_colloc[t] = co;
  }
  if constexpr (QOp::kNodalField) {
    // reference gradient of the cached nodal field (read plain: constrained
    // entries as stored), mf_nh_operator.h:873-877
    Number wg[3][3];
    evaluate_g<N, 3, Number, kRolled>(T, s_shape, s_colloc, w.v, wg);
    qop.attach(qd, wg);
  }

  Number val[NC], grad[NC][3];
  evaluate_vg<N, NC, Number, kRolled>(T, s_shape, s_colloc, u, val, grad);
  apply_qop(qop, cd, qd, val, grad);
  Number out[NC];
  integrate_vg<N, NC, Number, kSpareSlots, kRolled>(T, s_shape, s_colloc, val, grad, out);
  if constexpr (kToCells) {
    if (active) store_node<Number, NC>(dst + (int64_t)slot * NC, out);
    return;
  }
  if constexpr (kLateDst) {
    const NodeValues<Number, NC> v =
        active && !first ? load_node<Number, NC>(dst + node * NC) : NodeValues<Number, NC>{};
#pragma unroll
    for (int c = 0; c < NC; ++c) dold[c] = v.v[c];
  }
  if (active) {
    Number r[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) r[c] = dold[c] + out[c];
    if (((entry >> kConstraintShift) & ((1u << NC) - 1u)) == 0u) {
      store_node<Number, NC>(dst + node * NC, r);  // no constrained component: one wide store
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (!((entry >> (kConstraintShift + c)) & 1u)) dst[node * NC + c] = r[c];
    }
  }
}

// Spare tile slots (5 NC instead of 3 NC per cell, two barriers fewer per
// cell) where the larger tile stays within 16 KB per workgroup.
template <int P, int CPB, typename Number, int NC>
constexpr bool spare_slots() {
  return CPB * 5 * NC * (P + 1) * (P + 1) * (P + 1) * (int)sizeof(Number) <= 16384;
}

template <int P, int CPB, typename Number, class QOp>
__global__ void __launch_bounds__((block_threads<P, CPB>()))
    apply_cells(ApplyArgs<Number> a, QOp qop, int assign) {
  constexpr int N = P + 1, N3 = N * N * N, NC = QOp::NC, NT = block_threads<P, CPB>();
  constexpr bool kSpare = spare_slots<P, CPB, Number, NC>();
  __shared__ Number s_shape[N * N], s_colloc[N * N];
  __shared__ Number s_tile[CPB * (kSpare ? 5 : 3) * NC * N3];
  const int t = threadIdx.x;
  const int first_cell = a.cell_begin + xcd_remap(blockIdx.x, gridDim.x) * CPB;
  cell_group<P, Number, QOp, false, kSpare>(qop, a.cell_nodes, a.src, a.dst, first_cell, a.cell_end, CPB, assign,
                                            a.shape, a.colloc, s_shape, s_colloc, s_tile);
  // rows of constrained dofs: identity (mf_nh_operator.h:622-624).  The
  // cells never store a constrained component, so these rows can follow them.
  if (a.fix_mode) {
    const int64_t g = (int64_t)blockIdx.x * NT + t;
    for (int64_t idx = g; idx < a.n_constrained; idx += (int64_t)gridDim.x * NT) {
      const int64_t dof = a.constrained[idx];
      if (a.fix_mode == 1) a.dst[dof] = a.src[dof];
      else a.dst[dof] += a.src[dof];
    }
  }
}

// GATHER schedule, first launch: every cell at once, each point storing its
// contribution per cell (no colours, no read of dst).
template <int P, int CPB, typename Number, class QOp>
__global__ void __launch_bounds__((block_threads<P, CPB>()))
    apply_cells_to_cells(ApplyArgs<Number> a, QOp qop, Number *contrib) {
  constexpr int N = P + 1, N3 = N * N * N, NC = QOp::NC;
  constexpr bool kSpare = spare_slots<P, CPB, Number, NC>();  // as apply_cells: the same arithmetic
  __shared__ Number s_shape[N * N], s_colloc[N * N];
  __shared__ Number s_tile[CPB * (kSpare ? 5 : 3) * NC * N3];
  const int first_cell = a.cell_begin + xcd_remap(blockIdx.x, gridDim.x) * CPB;
  cell_group<P, Number, QOp, true, kSpare>(qop, a.cell_nodes, a.src, contrib, first_cell, a.cell_end, CPB, 1, a.shape,
                                           a.colloc, s_shape, s_colloc, s_tile, a.slots);
}

// GATHER schedule, second launch: one thread per node sums the contributions
// of its cells in colour order -- the order in which the colour launches add
// them, so the result is theirs bit for bit (up to the sign of a zero).
//
// A node's contributions are offsets[node] .. offsets[node + 1] in colour
// order.  With 3 components the first launch stores them at these places
// (index null): this launch then waits on two dependent loads and reads one
// contiguous stream.  A scalar field of low degree keeps them in point order
// (the 8-byte stores of its few points per cell would scatter) and this launch
// reads them through an index.  4 contributions are in flight at a time.
// Both launches together, against sums per component through an index in
// every case: solid Q4 FP64 0.2M unknowns 17.6 -> 11.9 us, 1M 45.5 -> 34.9;
// Q2 FP64 1.1M 77.9 -> 54.5 (FP32 49.8 -> 35.3); Q6 FP64 1.2M 66.5 -> 43.9;
// heat Q4 FP64 1M 47.5 -> 34.6.
template <typename Number, int NC>
__device__ inline void add_contributions(const Number *__restrict__ contrib, const uint32_t *__restrict__ index,
                                         int b, int e, Number (&acc)[NC]) {
  for (int k = b; k < e; k += 4) {
    NodeValues<Number, NC> v[4];
    uint32_t at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) at[u] = index && k + u < e ? index[k + u] : (uint32_t)(k + u);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < e) v[u] = load_node<Number, NC>(contrib + (int64_t)at[u] * NC);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + u < e)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = acc[c] + v[u].v[c];
  }
}

// What the sums of one operator read.
template <typename Number>
struct GatherTables {
  const Number *contrib;
  const int32_t *offsets;
  const uint32_t *index;  // or null: the contributions are in the nodes' order
  const uint8_t *cmask;   // constrained components of every node
};

template <typename Number>
inline GatherTables<Number> gather_tables(const OperatorData &op) {
  return GatherTables<Number>{op.contrib.as<Number>(), op.gather_offsets.as<int32_t>(),
                              op.gather_indexed ? op.gather_places.as<uint32_t>() : nullptr,
                              op.gather_cmask.as<uint8_t>()};
}

// The node's row of A src: the sum of its contributions, src itself on
// constrained components (identity rows).
template <typename Number, int NC>
__device__ inline void gather_row(const GatherTables<Number> &g, const Number *__restrict__ src, int64_t node,
                                  Number (&t)[NC]) {
  const int b = g.offsets[node], e = g.offsets[node + 1];
  const unsigned m = g.cmask[node];
  const NodeValues<Number, NC> f = load_node<Number, NC>(g.contrib + (int64_t)(g.index ? g.index[b] : b) * NC);
#pragma unroll
  for (int c = 0; c < NC; ++c) t[c] = f.v[c];
  add_contributions<Number, NC>(g.contrib, g.index, b + 1, e, t);
  if (m) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if ((m >> c) & 1u) t[c] = src[node * NC + c];
  }
}

// fix_mode 1 (vmult): dst = A src; 2 (vmult_add): dst += A src
template <typename Number, int NC>
__device__ inline void gather_node(const GatherTables<Number> &g, const Number *__restrict__ src,
                                   Number *__restrict__ dst, int64_t node, int fix_mode) {
  Number t[NC];
  if (fix_mode == 1) {
    gather_row<Number, NC>(g, src, node, t);
  } else {
    const int b = g.offsets[node], e = g.offsets[node + 1];
    const unsigned m = g.cmask[node];
    const NodeValues<Number, NC> o = load_node<Number, NC>(dst + node * NC);
#pragma unroll
    for (int c = 0; c < NC; ++c) t[c] = o.v[c];
    add_contributions<Number, NC>(g.contrib, g.index, b, e, t);
    if (m) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if ((m >> c) & 1u) t[c] = o.v[c] + src[node * NC + c];
    }
  }
  store_node<Number, NC>(dst + node * NC, t);
}

// small workgroups: a level of a few thousand nodes still spreads over the chip
constexpr int kGatherThreads = 64;

template <typename Number, int NC>
__global__ void __launch_bounds__(kGatherThreads)
    gather_contributions(GatherTables<Number> g, const Number *__restrict__ src, Number *__restrict__ dst,
                         int64_t n_nodes, int fix_mode) {
  const int64_t node = (int64_t)blockIdx.x * kGatherThreads + threadIdx.x;
  if (node >= n_nodes) return;
  gather_node<Number, NC>(g, src, dst, node, fix_mode);
}

// The sums with an epilogue: the row t of A x goes straight into the smoother's
// update (or the residual) with the expressions of the separate vector kernels,
// so the result is theirs bit for bit.  One launch and one store and load of t
// less per application.  With the restriction in two launches and no copies of
// the finest level's vectors: V-cycle of 64x16x16 Q4 cells FP64 2.11 -> 1.67
// ms, mixed MG-CG of 48x12x12 Q2 cells 2.75 -> 2.20 ms.
template <typename Number, int NC, int KIND>
__global__ void __launch_bounds__(kGatherThreads)
    gather_epilogue(GatherTables<Number> g, Number *x, const Number *__restrict__ b,
                    const Number *__restrict__ inv_diag, Number *__restrict__ d, Number *__restrict__ out, double s0,
                    double s1, int64_t n_nodes) {
  const int64_t node = (int64_t)blockIdx.x * kGatherThreads + threadIdx.x;
  if (node >= n_nodes) return;
  using Node = NodeValues<Number, NC>;
  const Node bv = load_node<Number, NC>(b + node * NC);
  Node iv{}, dv{}, xv{};
  if constexpr (KIND != kEpiResidual) {
    iv = load_node<Number, NC>(inv_diag + node * NC);
    xv = load_node<Number, NC>(x + node * NC);
  }
  if constexpr (KIND == kEpiChebUpdate) dv = load_node<Number, NC>(d + node * NC);
  Number t[NC], r[NC], v[NC];
  gather_row<Number, NC>(g, x, node, t);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if constexpr (KIND == kEpiResidual) {
      r[c] = bv.v[c] - t[c];
    } else {
      v[c] = KIND == kEpiChebFirstStep ? cheb_first_step_value<Number>(iv.v[c], bv.v[c], t[c], s0)
                                       : cheb_update_value<Number>(dv.v[c], iv.v[c], bv.v[c], t[c], s0, s1);
      r[c] = xv.v[c] + v[c];
    }
  }
  if constexpr (KIND == kEpiResidual) {
    store_node<Number, NC>(out + node * NC, r);
  } else {
    store_node<Number, NC>(d + node * NC, v);
    store_node<Number, NC>(x + node * NC, r);
  }
}

}  // namespace mfg
