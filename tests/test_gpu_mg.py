"""Device multigrid parity through the C ABI: transfer operators, one V-cycle,
Chebyshev eigenvalue estimates and MG-CG against the oracle on identical
hierarchies.  Bars: transfers and the V-cycle to 1e-12 / 1e-10 relative;
MG-CG solution within 1e-8 of the oracle's and iteration count within +-1."""
import numpy as np
import pytest
import torch

import mfgpu
import oracle as O

pytestmark = pytest.mark.gpu


def dev(x, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device="cuda", dtype=dtype)


def rel(a, b):
    a = a.detach().double().cpu().numpy() if hasattr(a, "detach") else a
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def hierarchy(kind, lo, hi, coarse, n_levels, p, precisions=None, face_mask=1, amp=1e-3, noise=1e-5,
              storage=mfgpu.T2_FOLDED):
    """Matching device and oracle hierarchies, linearised at interpolated u0;
    FP64 solid levels keep the given tensor2 point storage."""
    nc = 3 if kind == "solid" else 1
    cm = 7 if nc == 3 else 1
    precisions = precisions or [mfgpu.FP64] * n_levels
    gms = [mfgpu.BoxMesh(lo, hi, [c << l for c in coarse], p, nc, face_mask, cm) for l in range(n_levels)]
    oms = O.box_levels(lo, hi, coarse, n_levels, p, nc, face_mask, cm)
    if kind == "solid":
        gops = [mfgpu.NeoHookOperator(m, O.MU, O.NU, O.RHO, O.ALPHA1, precision=pr) for m, pr in zip(gms, precisions)]
        for op, pr in zip(gops, precisions):
            if pr == mfgpu.FP64:
                op.set_point_storage(storage)
        oops = [O.Solid(m, caching=1) for m in oms]
    else:
        gops = [mfgpu.LaplaceOperator(m, 0.1, None, precision=pr) for m, pr in zip(gms, precisions)]
        oops = [O.Heat(m, dt=0.1) for m in oms]
    trs = [mfgpu.Transfer(gops[l - 1], gops[l], mfgpu.box_children(gms[l - 1], gms[l])) for l in range(1, n_levels)]
    if kind == "solid":
        u = oms[-1].u0(amp=amp, noise=noise)
        us = [u]
        for l in range(n_levels - 1, 0, -1):
            us.insert(0, O.interpolate(oms[l - 1], oms[l], us[0]))
        for op, uu in zip(oops, us):
            op.cache(uu)
        # interpolate_to_mg on the device, each level in its own precision
        ug = [None] * n_levels
        ug[-1] = dev(u, gops[-1].dtype)
        for l in range(n_levels - 1, 0, -1):
            ug[l - 1] = torch.empty(gms[l - 1].n_dofs, dtype=gops[l - 1].dtype, device="cuda")
            trs[l - 1].interpolate(ug[l - 1], ug[l])
        for op, uu in zip(gops, ug):
            op.cache(uu)
    return gms, oms, gops, oops, trs


@pytest.mark.parametrize("p,nc", [(1, 3), (2, 1), (2, 3), (4, 3)])
def test_transfer_parity(cuda, p, nc):
    kind = "solid" if nc == 3 else "heat"
    gms, oms, gops, oops, trs = hierarchy(kind, [0, 0, 0], [2.0, 1.0, 1.0], [2, 1, 1], 2, p, face_mask=1 | 16)
    cm, fm = oms
    c = O.fill_uniform(11, cm.n_dofs)
    f = O.fill_uniform(12, fm.n_dofs)
    fo = f.copy()
    O.prolongate_add(cm, fm, c, fo)
    fg = dev(f)
    trs[0].prolongate_add(fg, dev(c))
    assert rel(fg, fo) < 1e-13
    co = c.copy()
    O.restrict_add(cm, fm, f, co)
    cg = dev(c)
    trs[0].restrict_add(cg, dev(f))
    assert rel(cg, co) < 1e-13
    ci = torch.empty(cm.n_dofs, dtype=torch.float64, device="cuda")
    trs[0].interpolate(ci, dev(f))
    assert rel(ci, O.interpolate(cm, fm, f)) < 1e-13


@pytest.mark.parametrize("precisions", [(mfgpu.FP64, mfgpu.FP64), (mfgpu.FP64, mfgpu.FP32), (mfgpu.FP32, mfgpu.FP32)])
@pytest.mark.parametrize("p,nc", [(1, 1), (3, 3), (5, 3), (6, 3), (5, 1), (6, 1)])
def test_transfers_by_degree(cuda, p, nc, precisions):
    """The degrees whose kernels take one or all components at a time, in every
    pair of level precisions."""
    print(f"transfers p={p} nc={nc} precisions={precisions}", flush=True)
    cmask = 7 if nc == 3 else 1
    gms = [mfgpu.BoxMesh([0, 0, 0], [2.0, 1.0, 1.0], n, p, nc, 1 | 16, cmask) for n in ([3, 1, 2], [6, 2, 4])]
    cm, fm = O.box_levels([0, 0, 0], [2.0, 1.0, 1.0], [3, 1, 2], 2, p, nc, 1 | 16, cmask)
    ops = [mfgpu.NeoHookOperator(m, O.MU, O.NU, O.RHO, O.ALPHA1, precision=q) if nc == 3
           else mfgpu.LaplaceOperator(m, 0.1, None, precision=q) for m, q in zip(gms, precisions)]
    t = mfgpu.Transfer(ops[0], ops[1], mfgpu.box_children(gms[0], gms[1]))
    c, f = O.fill_uniform(11, cm.n_dofs), O.fill_uniform(12, fm.n_dofs)
    c, f = (v.astype(np.float32).astype(np.float64) for v in (c, f))  # exact in every precision
    fo, co = f.copy(), c.copy()
    O.prolongate_add(cm, fm, c, fo)
    O.restrict_add(cm, fm, f, co)
    fg, cg = dev(f, ops[1].dtype), dev(c, ops[0].dtype)
    t.prolongate_add(fg, dev(c, ops[0].dtype))
    t.restrict_add(cg, dev(f, ops[1].dtype))
    # sums in 64 bits, stored once (prolongation) or after each of up to 8 cells
    eps = [1e-13 if q == mfgpu.FP64 else 8 * 2.0 ** -24 for q in precisions]
    assert rel(fg, fo) < eps[1] and rel(cg, co) < eps[0]


def test_vcycle_and_eigenvalues_small_config(cuda):
    """8^3 Q2 cube, 3 levels, Chebyshev degree 4 (FP64 levels)."""
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [1, 1, 1], [2, 2, 2], 3, 2)
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30)
    mg.setup()
    src = O.fill_uniform(5, oms[-1].n_dofs)
    ref, eig = O.mg_vmult(oms, oops, src, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30)
    for l in range(3):
        lmax, lmin, deg = mg.level_info(l)
        assert abs(lmax - eig[l][0]) < 1e-9 * eig[l][0], (l, lmax, eig[l])
        assert deg == int(eig[l][2])
    dst = torch.empty_like(dev(src))
    mg.vmult(dst, dev(src))
    assert rel(dst, ref) < 1e-9


@pytest.mark.parametrize("coarse_kind", [0, 1])
def test_mg_cg_small_config(cuda, coarse_kind):
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [1, 1, 1], [2, 2, 2], 3, 2)
    fine, A = oms[-1], oops[-1]
    xt = O.fill_uniform(2, fine.n_dofs)
    xt[fine.constrained()] = 0.0
    b = A.vmult(xt)
    xo, it_o, rel_o = O.mg_cg_solve(oms, oops, b, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30,
                                    coarse_kind=coarse_kind, tol_rel=1e-8)
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30,
                         coarse_kind=coarse_kind, coarse_tolerance=1e-3)
    mg.setup()
    x = torch.zeros(fine.n_dofs, dtype=torch.float64, device="cuda")
    info = mfgpu.cg_solve(gops[-1], dev(b), x, mfgpu.PRECOND_MG, mg, tol_rel=1e-8)
    print(f"coarse_kind={coarse_kind}: iterations gpu {info.iterations} oracle {it_o}")
    assert abs(info.iterations - it_o) <= 1
    assert info.final_residual <= 1e-8 * np.linalg.norm(b)
    assert rel(x, xo) < 1e-8
    assert rel(x, xt) < 1e-6


def test_mg_cg_gradient_storage(cuda):
    """MG-CG with every level in the 10-word tensor2 storage: the oracle's
    iteration count (+-1) and solution, as with the folded storage."""
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [1, 1, 1], [2, 2, 2], 3, 2, storage=mfgpu.T2_GRADIENT)
    assert all(op.n_fields() == 10 for op in gops)
    fine, A = oms[-1], oops[-1]
    xt = O.fill_uniform(2, fine.n_dofs)
    xt[fine.constrained()] = 0.0
    b = A.vmult(xt)
    xo, it_o, rel_o = O.mg_cg_solve(oms, oops, b, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30,
                                    coarse_kind=0, tol_rel=1e-8)
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30, coarse_kind=0,
                         coarse_tolerance=1e-3)
    mg.setup()
    x = torch.zeros(fine.n_dofs, dtype=torch.float64, device="cuda")
    info = mfgpu.cg_solve(gops[-1], dev(b), x, mfgpu.PRECOND_MG, mg, tol_rel=1e-8)
    assert abs(info.iterations - it_o) <= 1
    assert rel(x, xo) < 1e-8
    assert rel(x, xt) < 1e-6


def test_jacobi_and_plain_cg(cuda):
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [1, 1, 1], [4, 4, 4], 1, 2)
    A, G = oops[0], gops[0]
    b = A.vmult(O.fill_uniform(3, oms[0].n_dofs))
    G.compute_diagonal()
    for pre in (0, 1):
        xo, it_o, _ = O.cg_solve(A, b, precond=pre, omega=0.65, tol_rel=1e-8)
        x = torch.zeros_like(dev(b))
        info = mfgpu.cg_solve(G, dev(b), x, pre, None, omega=0.65, tol_rel=1e-8)
        assert abs(info.iterations - it_o) <= 1, (pre, info.iterations, it_o)
        assert rel(x, xo) < 1e-7
    with pytest.raises(mfgpu.MfgError) as e:
        mfgpu.cg_solve(G, dev(b), torch.zeros_like(dev(b)), 0, None, tol_rel=1e-12, max_iter=3)
    assert e.value.code == 4


def test_heat_mg_cg(cuda):
    gms, oms, gops, oops, trs = hierarchy("heat", [0, 0, 0], [1, 1, 1], [2, 2, 2], 3, 3, face_mask=63)
    fine, A = oms[-1], oops[-1]
    xt = O.fill_uniform(2, fine.n_dofs)
    xt[fine.constrained()] = 0.0
    b = A.vmult(xt)
    xo, it_o, _ = O.mg_cg_solve(oms, oops, b, cheb_degree=5, smoothing_range=15.0, eig_cg_iterations=10,
                                tol_rel=1e-10)
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=5, smoothing_range=15.0, eig_cg_iterations=10)
    mg.setup()
    x = torch.zeros(fine.n_dofs, dtype=torch.float64, device="cuda")
    info = mfgpu.cg_solve(gops[-1], dev(b), x, mfgpu.PRECOND_MG, mg, tol_rel=1e-10)
    assert abs(info.iterations - it_o) <= 1
    assert rel(x, xt) < 1e-8


def test_mixed_precision_mg_cg(cuda):
    """FP32 V-cycle (levels 1.., caches from FP32 u), FP64 coarse level and
    outer CG: reaches the FP64 residual 1e-8; solution within the solver
    tolerance of the FP64-preconditioned solve."""
    prec = [mfgpu.FP64, mfgpu.FP32, mfgpu.FP32]
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [1, 1, 1], [2, 2, 2], 3, 2, precisions=prec)
    fine_op64 = mfgpu.NeoHookOperator(gms[-1], O.MU, O.NU, O.RHO, O.ALPHA1)
    u = oms[-1].u0(amp=1e-3, noise=1e-5)
    fine_op64.cache(dev(u))
    xt = O.fill_uniform(2, oms[-1].n_dofs)
    xt[oms[-1].constrained()] = 0.0
    b = oops[-1].vmult(xt)
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=4, smoothing_range=20.0, eig_cg_iterations=30, coarse_kind=1)
    mg.setup()
    x = torch.zeros(oms[-1].n_dofs, dtype=torch.float64, device="cuda")
    info = mfgpu.cg_solve(fine_op64, dev(b), x, mfgpu.PRECOND_MG, mg, tol_rel=1e-8)
    assert info.final_residual <= 1e-8 * np.linalg.norm(b)
    xo, it_o, _ = O.mg_cg_solve(oms, oops, b, cheb_degree=4, tol_rel=1e-8, coarse_kind=1)
    print(f"mixed: iterations {info.iterations} (fp64 oracle {it_o}), err vs fp64 solve {rel(x, xo):.2e}")
    assert info.iterations <= it_o + 3
    assert rel(x, xo) < 1e-6


@pytest.mark.parametrize("coarse_kind,precisions", [(1, None), (0, None), (1, [mfgpu.FP64, mfgpu.FP32, mfgpu.FP32])])
def test_graphed_vcycle_equals_eager(cuda, coarse_kind, precisions):
    """The V-cycle's sweeps replayed as hipGraphs give bitwise the eager
    results: over several replays with eager work in between, after a new
    linearisation (re-setup and re-capture), and through MG-CG."""
    print(f"graphed V-cycle coarse_kind={coarse_kind} precisions={precisions}", flush=True)
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [2.0, 1.0, 1.0], [2, 1, 1], 3, 3, precisions=precisions)
    eager = mfgpu.Multigrid(gops, trs, cheb_degree=5, coarse_kind=coarse_kind)
    graphed = mfgpu.Multigrid(gops, trs, cheb_degree=5, coarse_kind=coarse_kind)
    eager.use_graph(False)
    graphed.use_graph(True)
    n = gms[-1].n_dofs
    for relinearised in (False, True):
        if relinearised:
            for op, m in zip(gops, gms):  # another linearisation point on every level
                op.cache(dev(m.u0(amp=2e-3, noise=1e-5, seed=9), op.dtype))
        eager.setup()
        graphed.setup()
        for rep in range(4):
            src = mfgpu.fill_uniform(20 + rep, torch.empty(n, dtype=torch.float64, device="cuda"))
            want = torch.empty_like(src)
            got = torch.full_like(src, float("nan"))
            eager.vmult(want, src)
            graphed.vmult(got, src)
            assert torch.equal(got, want), (relinearised, rep)
            torch.cuda.synchronize()
            _ = float(src.sum())  # eager work between replays
        assert graphed.graph_nodes() > 0 and eager.graph_nodes() == 0
    fine = gops[-1] if precisions is None else mfgpu.NeoHookOperator(gms[-1], O.MU, O.NU, O.RHO, O.ALPHA1)
    if precisions is not None:
        fine.cache(dev(gms[-1].u0(amp=2e-3, noise=1e-5, seed=9)))
    b = mfgpu.fill_uniform(30, torch.empty(n, dtype=torch.float64, device="cuda"))
    x1, x2 = torch.zeros_like(b), torch.zeros_like(b)
    i1 = mfgpu.cg_solve(fine, b, x1, mfgpu.PRECOND_MG, eager, tol_rel=1e-8)
    i2 = mfgpu.cg_solve(fine, b, x2, mfgpu.PRECOND_MG, graphed, tol_rel=1e-8)
    assert i1.iterations == i2.iterations and torch.equal(x1, x2)


def test_coarse_cg_results_independent_of_history(cuda):
    """The V-cycle's coarse CG stops on the device and the host reads its
    state after runs of iterations sized by the previous coarse solve: the
    results must not depend on that history.  The same input gives bitwise the
    same output after another input (another coarse residual history) and on a
    fresh hierarchy whose first coarse solve reads back after one iteration."""
    print("coarse CG history independence", flush=True)
    gms, oms, gops, oops, trs = hierarchy("solid", [0, 0, 0], [2.0, 1.0, 1.0], [2, 1, 1], 3, 3)
    n = gms[-1].n_dofs
    x = mfgpu.fill_uniform(40, torch.empty(n, dtype=torch.float64, device="cuda"))
    y = torch.zeros_like(x)
    y[n // 3] = 1.0  # a point load
    mg = mfgpu.Multigrid(gops, trs, cheb_degree=5, coarse_kind=1, coarse_tolerance=1e-6)
    mg.setup()
    outs = []
    for src in (x, y, x, y, x):
        out = torch.full_like(src, float("nan"))
        mg.vmult(out, src)
        outs.append(out)
    fresh = mfgpu.Multigrid(gops, trs, cheb_degree=5, coarse_kind=1, coarse_tolerance=1e-6)
    fresh.setup()
    first = torch.full_like(x, float("nan"))
    fresh.vmult(first, x)
    assert torch.isfinite(outs[0]).all() and torch.isfinite(outs[1]).all()
    assert torch.equal(outs[0], outs[2]) and torch.equal(outs[0], outs[4]) and torch.equal(outs[0], first)
    assert torch.equal(outs[1], outs[3])


@pytest.mark.parametrize("kind,p,n,precision", [
    ("solid", 1, (4, 6, 2), mfgpu.FP64), ("solid", 2, (6, 4, 4), mfgpu.FP32), ("solid", 4, (4, 4, 2), mfgpu.FP64),
    ("solid", 5, (2, 4, 2), mfgpu.FP32), ("solid", 6, (4, 2, 2), mfgpu.FP64), ("heat", 1, (8, 6, 4), mfgpu.FP64),
    ("heat", 2, (6, 6, 2), mfgpu.FP32), ("heat", 3, (4, 4, 4), mfgpu.FP64), ("heat", 6, (4, 2, 2), mfgpu.FP32)])
def test_vcycle_gather_equals_colours(cuda, kind, p, n, precision):
    """The V-cycle with the smoother's updates and the residual inside the
    per-node sums, the restriction in two launches and the caller's vectors as
    the finest level's is bitwise the one of colour launches, separate vector
    passes and copies; so it is from another precision, and in place."""
    print(f"V-cycle gather = colours {kind} p={p} precision={precision}", flush=True)
    out = {}
    for sched in (None, mfgpu.CELLS_COLOURS):
        inst = mfgpu.Instance(kind, n, p, level_precision=precision, seed=3, cell_schedule=sched,
                              coarse_eig_iterations=40)
        dt = inst.levels[-1].dtype
        x = mfgpu.fill_uniform(11, torch.empty(inst.n_dofs, dtype=dt, device="cuda"))
        y = torch.full_like(x, float("nan"))
        keep = x.clone()
        inst.mg.vmult(y, x)
        other = torch.float32 if dt == torch.float64 else torch.float64
        z = torch.empty(inst.n_dofs, dtype=other, device="cuda")
        inst.mg.vmult(z, x.to(other))
        w = x.clone()  # in place, through the C interface
        mfgpu.check(mfgpu.lib().mfg_mg_vmult(inst.mg.h, mfgpu._ptr(w), mfgpu._ptr(w),
                                             mfgpu.FP64 if dt == torch.float64 else mfgpu.FP32))
        assert torch.equal(x, keep) and torch.isfinite(y).all() and torch.equal(w, y)
        out[sched] = (y, z)
    a, b = out[None], out[mfgpu.CELLS_COLOURS]
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("kind,p,n,precision", [
    ("solid", 2, (36, 36, 34), mfgpu.FP64), ("solid", 4, (22, 22, 20), mfgpu.FP32), ("heat", 2, (36, 36, 34), mfgpu.FP32),
    ("heat", 4, (22, 22, 20), mfgpu.FP64)])
def test_vcycle_gather_inside_a_hierarchy(cuda, kind, p, n, precision):
    """Above 2^20 points an operator applies itself by colours and a hierarchy
    applies it with GATHER: estimates, diagonals and V-cycles are bitwise those of
    a hierarchy whose operators were set to COLOURS, before and after the schedule
    is set on a hierarchy in use, and the operator's own vmult stays as it was."""
    print(f"GATHER inside a hierarchy {kind} p={p} precision={precision}", flush=True)
    assert 2 ** 20 < n[0] * n[1] * n[2] * (p + 1) ** 3 <= 3 * 2 ** 20
    out = []
    for sched in (None, mfgpu.CELLS_COLOURS):
        inst = mfgpu.Instance(kind, n, p, level_precision=precision, seed=3, cell_schedule=sched, coarse_eig_iterations=20)
        top = inst.levels[-1]
        assert top.cell_schedule() == mfgpu.CELLS_COLOURS
        x = mfgpu.fill_uniform(11, torch.empty(inst.n_dofs, dtype=top.dtype, device="cuda"))
        y, z, w = (torch.full_like(x, float("nan")) for _ in range(3))
        inst.mg.vmult(y, x)
        top.vmult(z, x)
        info = [inst.mg.level_info(l) for l in range(len(inst.levels))]
        top.compute_diagonal()
        out.append((y, z, top.diagonal(), info))
        if sched is None:
            top.set_cell_schedule(mfgpu.CELLS_COLOURS)
            inst.mg.vmult(w, x)
            assert torch.equal(w, y)
    assert torch.isfinite(out[0][0]).all() and out[0][3] == out[1][3]
    assert all(torch.equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))


@pytest.mark.parametrize("kind,p,n,precision", [("solid", 2, (4, 4, 2), mfgpu.FP64), ("heat", 3, (4, 2, 4), mfgpu.FP32),
                                                ("heat", 2, (3, 3, 3), mfgpu.FP64)])
@pytest.mark.parametrize("graph", [False, True])
def test_vcycle_overlapping_vectors(cuda, kind, p, n, precision, graph):
    """src and dst may be views that share a part of their memory: the V-cycle is
    the one of separate vectors, whichever of them comes first.  The third case
    has one level."""
    print(f"V-cycle of overlapping vectors {kind} p={p} precision={precision} graph={graph}", flush=True)
    inst = mfgpu.Instance(kind, n, p, level_precision=precision, seed=3, coarse_eig_iterations=40)
    inst.mg.use_graph(graph)
    m, dt = inst.n_dofs, inst.levels[-1].dtype
    x = mfgpu.fill_uniform(11, torch.empty(m, dtype=dt, device="cuda"))
    y = torch.empty_like(x)
    inst.mg.vmult(y, x)
    for src_at, dst_at in ((0, 1), (1, 0), (0, m // 2), (m - 1, 0), (0, m), (m, 0)):
        buf = torch.full((2 * m,), float("nan"), dtype=dt, device="cuda")
        src, dst = buf[src_at:src_at + m], buf[dst_at:dst_at + m]
        src.copy_(x)
        mfgpu.check(mfgpu.lib().mfg_mg_vmult(inst.mg.h, mfgpu._ptr(dst), mfgpu._ptr(src), precision))
        assert torch.equal(dst, y), (src_at, dst_at)


@pytest.mark.parametrize("kind,p,n", [("solid", 1, (1, 1, 1)), ("solid", 1, (6, 2, 3)), ("solid", 2, (2, 1, 2)),
                                      ("heat", 1, (7, 7, 4)), ("heat", 2, (3, 3, 3))])
def test_eigenvalue_estimate_small_levels(cuda, kind, p, n):
    """The fixed-count CG's estimate on levels of one to two workgroups of
    unknowns, run until it stops by itself (||r|| <= 1e-15 ||r_0||; the remaining
    iterations change nothing), against the oracle's."""
    print(f"eigenvalue estimate {kind} p={p} n={n}", flush=True)
    nc, fm, cm = (3, 1, 7) if kind == "solid" else (1, 63, 1)
    lo, hi = [0, 0, 0], [1.0, 0.7, 0.5]
    gm, om = mfgpu.BoxMesh(lo, hi, list(n), p, nc, fm, cm), O.Mesh(lo, hi, list(n), p, nc, fm, cm)
    if kind == "solid":
        u = om.u0(amp=1e-2, noise=1e-5)
        op, oo = mfgpu.NeoHookOperator(gm, O.MU, O.NU, O.RHO, O.ALPHA1), O.Solid(om, caching=1)
        op.cache(dev(u))
        oo.cache(u)
    else:
        op, oo = mfgpu.LaplaceOperator(gm, 0.1, None), O.Heat(om, dt=0.1, coef=np.ones(om.n_cells * (p + 1) ** 3))
    mg = mfgpu.Multigrid([op], [], coarse_eig_iterations=gm.n_dofs)
    mg.setup()
    # an extreme Lanczos value is stable to rounding until the run stops
    lmax = O.cheb_eigenvalues(oo, gm.n_dofs)[0]
    assert abs(mg.level_info(0)[0] - lmax) <= 1e-8 * lmax
