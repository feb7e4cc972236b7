// Device operator object shared by the operator, multigrid and solver code.
#pragma once
#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace mfg {

// Operators with at most this many quadrature points use the GATHER schedule by
// default: two launches over all cells against 8 of one colour each, whose
// cells alone do not fill the GPU.  The contribution buffer is one per
// operator, so a larger default would add a buffer that two applications on
// different streams (set_stream in between) share.
constexpr int64_t kGatherMaxPoints = 1 << 20;
// Where the operator's work is ordered on one stream (multigrid levels, the
// operators of a SolidProblem), GATHER serves up to this many points.  Past it
// the colours' plain read-modify-write moves less than the contributions'
// store and load.  Measured, time of colours / gather on cubes: solid Q1 1.3
// at 0.55M points, 0.77 at 2.6M; Q2 1.23 at 1.2M, 1.02 at 3.4M, 0.84 at 6.8M;
// Q3 1.47 at 0.9M, 1.07 at 2.3M, 0.94 at 4.7M; Q4 1.55 at 0.6M, 1.07 at 3.7M,
// 0.88 at 8M (FP32 1.00); Q5 1.10 at 3.4M; Q6 1.39 at 3.2M, 1.15 at 6M; heat
// Q2 0.96 at 3.4M (FP32 1.40), Q3 1.22 at 2.3M, Q4 1.04 at 5.8M, Q6 1.31 at
// 4.7M.  One limit per degree for both kinds and precisions: about where the
// first of them stops gaining, and leaves what others would gain above it.
constexpr int64_t gather_max_points(int p) {
  return p == 1 ? kGatherMaxPoints : p <= 3 ? 3 * kGatherMaxPoints : 5 * kGatherMaxPoints;
}

// device bytes of the GATHER schedule's tables and contribution buffer
inline size_t gather_bytes(int64_t nqp, int64_t n_nodes, int nc, size_t es) {
  return (size_t)nqp * (nc * es + 4) + (size_t)(n_nodes + 1) * 4 + (size_t)n_nodes;
}

// Whether the trilinear map of a cell (8 vertices, vertex v at (v & 1, v >> 1 & 1,
// v >> 2 & 1)) is affine: its mixed terms vanish.
inline bool affine_cell(const double *X) {
  auto V = [&](int v, int e) { return X[v * 3 + e]; };
  double h = 0, mixed = 0;
  for (int e = 0; e < 3; ++e) {
    for (int v : {1, 2, 4}) h = std::max(h, std::fabs(V(v, e) - V(0, e)));
    mixed = std::max({mixed, std::fabs(V(3, e) - V(2, e) - V(1, e) + V(0, e)),
                      std::fabs(V(5, e) - V(4, e) - V(1, e) + V(0, e)),
                      std::fabs(V(6, e) - V(4, e) - V(2, e) + V(0, e)),
                      std::fabs(V(7, e) - V(6, e) - V(5, e) + V(4, e) - V(3, e) + V(2, e) + V(1, e) - V(0, e))});
  }
  return mixed <= 1e-12 * h;
}

// What the per-node sums of a GATHER application do with a row t of A x
// besides storing it: the pass that would follow over the same vectors.
enum GatherEpilogue : int {
  kEpiResidual = 0,   // out = b - t
  kEpiChebFirstStep,  // d = D^{-1} (b - t) s0; x += d
  kEpiChebUpdate,     // d = s0 d + s1 D^{-1} (b - t); x += d
};
struct EpilogueArgs {
  int kind;
  const void *b;
  void *out;  // residual
  void *d;    // Chebyshev direction
  double s0, s1;
};

struct OperatorData {
  int kind = 0;  // 0 solid (NeoHookOperator), 1 heat (LaplaceOperator)
  int precision = MFG_FP64;
  int p = 1, nc = 1, n_cells = 0, n_fields = 0;
  int64_t n_nodes = 0, n_dofs = 0, nqp = 0, n_constrained = 0;
  hipStream_t stream = nullptr;
  mfg_solid_params sp{};
  double kappa = 0, c_1 = 0, lambda = 0, rho_alpha = 0, dt = 0;  // material 0
  // neo-Hookean constants (material.h:78-94) of material 0 and of the
  // inclusion material, used on cells whose material id is not 0
  // (mf_nh_operator.h:404, 656-658)
  struct MaterialConstants {
    double mu = 0, lambda = 0, kappa = 0, c_1 = 0, rho = 0, rho_alpha = 0;
  };
  MaterialConstants mats[2];
  bool ready = false, has_diagonal = false;

  DeviceBuffer cell_nodes;   // uint32: node | constraint bits << 28
  DeviceBuffer constrained;  // int32 sorted dof list
  DeviceBuffer vertices;     // double n_cells*24
  DeviceBuffer tab_shape, tab_colloc, tab_sq, tab_points, tab_weights;
  DeviceBuffer qd;           // quadrature cache, field-major SoA
  DeviceBuffer diag, inv_diag;
  DeviceBuffer u_nodal;      // the linearisation point (scalar_referential caching)
  // the linearisation point of the 10-word storage, after its fields in qd
  template <class T>
  T *u_copy() const {
    return qd.as<T>() + (size_t)n_fields * nqp;
  }
  // reference-frame JxW per cell: when every cell's trilinear map is affine,
  // JxW_ref = cell_jxw[stored cell] * wq3[point] (tensor2, formulation 1)
  bool affine_ref = false;
  DeviceBuffer cell_jxw, wq3;
  DeviceBuffer cell_geo;  // heat on affine cells: Jinv Jinv^T (6, symmetric), det J per stored cell
  DeviceBuffer cell_met;  // solid on affine cells: J_ref^{-1} J_ref^{-T} (6, symmetric) per stored cell
  bool cartesian_ref = false;  // affine, and every cell's J_ref is diagonal
  int t2_storage = MFG_T2_FOLDED;  // tensor2 formulation-1 point storage (MFG_T2_*)
  bool t2_gradient() const { return kind == 0 && sp.caching == MFG_CACHING_TENSOR2 && sp.formulation == 1 && t2_storage == MFG_T2_GRADIENT; }
  // Error flag that the kernels of cache(), compute_diagonal() and the residual
  // set; these calls clear it, launch, synchronise and look at it.
  mutable PinnedHost<int> flag;
  int *clear_flag() const {
    flag.allocate();
    *flag.ptr = 0;
    return flag.ptr;
  }
  std::vector<int32_t> host_constrained;
  std::vector<int32_t> host_cell_nodes;  // input cell order (used to build transfers)
  std::vector<uint8_t> host_cmask;       // per node: constrained components
  // cells are stored colour-major: perm[c] = input index of stored cell c,
  // colour k occupies stored cells [colour_start[k], colour_start[k+1])
  std::vector<int32_t> perm;
  std::vector<int> colour_start;
  // with an inclusion material the cells of colour k are sorted by material
  // (as MatrixFree batches cells by cell_vectorization_category,
  // mf_elasticity.h:837-855): material 0 in [colour_start[k], mat_split[k]),
  // the inclusion in [mat_split[k], colour_start[k+1]).  Empty otherwise.
  std::vector<int> mat_split;
  bool has_inclusion() const { return !mat_split.empty(); }
  // f(colour, first stored cell, end, material) for every non-empty range of
  // one colour and one material, in launch (stored) order
  template <class F>
  void for_each_range(F f) const {
    for (size_t k = 0; k + 1 < colour_start.size(); ++k) {
      const int b = colour_start[k], e = colour_start[k + 1], s = has_inclusion() ? mat_split[k] : e;
      if (s > b) f((int)k, b, s, 0);
      if (e > s) f((int)k, s, e, 1);
    }
  }
  DeviceBuffer perm_dev;
  void colour_cells(const mfg_level_desc &d, int N3);
  int cell_schedule = MFG_CELLS_COLOURS;
  // bumped whenever a device buffer that apply() reads is reallocated (graphs
  // that captured the old addresses must be re-captured)
  uint64_t buffers_version = 0;
  // GATHER schedule: node v's contributions in colour order are entries
  // gather_offsets[v] .. gather_offsets[v + 1] of contrib, or (gather_indexed)
  // of the points listed in gather_places, contrib being in point order;
  // otherwise gather_places holds the place of every (stored cell, point).
  // cmask: the node's constrained components.
  DeviceBuffer gather_offsets, gather_places, gather_cmask, contrib;
  bool gather_indexed = false;
  // the contributions of the Newton residual and the diagonal (synchronous
  // calls: no two share it, and an application in flight on another stream has
  // its own), made by the first of them; false: no memory for it, and the call
  // takes the colour launches, which need none
  mutable DeviceBuffer setup_contrib;
  bool reserve_setup_contrib() const {
    const size_t need = (size_t)nqp * nc * elem_size();
    return setup_contrib.bytes >= need || setup_contrib.try_allocate(need);
  }
  const uint32_t *gather_slots() const { return gather_indexed ? nullptr : gather_places.as<uint32_t>(); }
  // All of the tables and the contribution buffer, or none of them.  Without
  // memory for them: MFG_ERR_HIP, or (optional) false.
  bool build_gather(bool optional = false);
  // The schedule was set through mfg_operator_set_cell_schedule: every
  // application keeps it.
  bool schedule_set = false;
  // Up to gather_max_points() a multigrid hierarchy (whose work, like its level
  // vectors, is ordered on one stream) applies its level operators with GATHER
  // whatever their default: prepare_gather() in its setup, apply_ordered() then.
  // Without memory for it they keep their default.
  void prepare_gather();
  bool gather_ordered() const { return cell_schedule == MFG_CELLS_GATHER || (!schedule_set && gather_ready); }
  bool gather_ready = false;
  // optional cell-kernel timing
  bool timing = false;
  mutable std::vector<std::pair<hipEvent_t, hipEvent_t>> events;
  mutable size_t events_used = 0;
  ~OperatorData();

  void setup_layout(const mfg_level_desc &d);
  void setup_solid();
  void setup_heat(const mfg_level_desc &d, const double *coef);
  void cache(const void *u, int u_precision);
  void export_qp_gradient(void *out);
  // dst (+)= A src on `on` (the operator's stream when null)
  void apply(const void *src, void *dst, bool add, hipStream_t on = nullptr) const;
  // dst = A src for callers that order all of the operator's work on its stream
  void apply_ordered(const void *src, void *dst) const;
  // where gather_ordered(): A x into the epilogue (the Chebyshev ones update x)
  void apply_epilogue(void *x, const EpilogueArgs &e) const;
  void compute_diagonal();
  size_t memory_consumption() const;
  // words per point of the quadrature cache of a solid operator
  static int solid_fields(const mfg_solid_params &sp, bool t2_gradient, bool affine);
  size_t elem_size() const { return precision == MFG_FP64 ? 8 : 4; }
  void timing_begin(hipStream_t s) const;
  void timing_end(hipStream_t s) const;
  void timing_collect(double &ms, int64_t &n);
};

}  // namespace mfg

struct mfg_operator_t : mfg::OperatorData {};
