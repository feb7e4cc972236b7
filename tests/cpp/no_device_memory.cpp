// What the optional buffers of the GATHER schedule do when the device refuses
// them: the operator, the transfer and the set-up calls stay with the colour
// launches, which need none.  Run where there is no GPU, so that every device
// allocation fails.
#include <cstdio>

#include "../../matrix-free-dealii-precice_amd/csrc/operator.hpp"
#include "../../matrix-free-dealii-precice_amd/csrc/solver.hpp"

static int check(bool ok, const char *what) {
  std::printf("%s: %s\n", what, ok ? "ok" : "FAILED");
  return ok ? 0 : 1;
}

int main() {
  using namespace mfg;
  void *p = nullptr;
  if (hipMalloc(&p, 8) == hipSuccess) {
    std::puts("a device is present");
    return 2;
  }
  int bad = 0;
  // one Q1 cell
  OperatorData op;
  op.p = 1;
  op.nc = 3;
  op.n_cells = 1;
  op.n_nodes = op.nqp = 8;
  op.n_dofs = 24;
  op.perm = {0};
  op.host_cell_nodes = {0, 1, 2, 3, 4, 5, 6, 7};
  op.host_cmask.assign(8, 0);
  try {
    op.prepare_gather();
    bad += check(!op.gather_ready && !op.gather_ordered() && !op.contrib.ptr && !op.gather_places.ptr &&
                     op.cell_schedule == MFG_CELLS_COLOURS,
                 "operator stays with the colours");
    bad += check(!op.reserve_setup_contrib() && op.setup_contrib.bytes == 0, "residual and diagonal stay with the colours");
  } catch (const Error &e) {
    bad += check(false, e.what());
  }
  bool refused = false;
  try {
    op.build_gather();  // the schedule asked for by name
  } catch (const Error &e) {
    refused = e.code == MFG_ERR_HIP;
  }
  bad += check(refused && !op.gather_offsets.ptr && !op.gather_places.ptr && !op.gather_cmask.ptr && !op.contrib.ptr,
               "an explicit GATHER schedule is refused and leaves nothing behind");
  TransferData t;
  t.coarse = &op;
  t.nc = 3;
  int tables = 0;
  op.gather_places.ptr = &tables;  // as if the tables were there
  try {
    t.prepare_restrict();
    bad += check(!t.contrib.ptr, "restriction stays with the colours");
  } catch (const Error &e) {
    bad += check(false, e.what());
  }
  op.gather_places.ptr = nullptr;
  if (!bad) std::puts("NO DEVICE MEMORY OK");
  return bad ? 1 : 0;
}
