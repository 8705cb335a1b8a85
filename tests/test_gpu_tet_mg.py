"""Geometric multigrid on tet4 meshes laid on a grid of cells (six tets per
cell, the jittered-grid meshes of the tet configuration): the Galerkin
hierarchy of the tet operator, against a direct solve and against the
Jacobi-preconditioned CG it replaces, and OC trajectories against the
oracle; at the configuration's size (100x50x50 cells, 1.5M tets, 788k DOF)
three OC iterations with the r = 1.5 filter and Emin = 1e-9 run with
property checks (true residual, energy identity, mixed vs fp64)."""
import numpy as np
import pytest

from oracle import driver as odrv
from oracle import fem as ofem
from oracle import problems as oprob
from oracle import transforms as tr

pytestmark = pytest.mark.gpu


def _tet_task(task_o, grid=True):
    from sktopt_amd import mesh as pmesh
    pm = task_o.mesh
    m = pmesh.MeshTet(pm.p, pm.t, cell_grid=pm.grid if grid else None)
    return pmesh.LinearElasticity(m, task_o.dirichlet_nodes, task_o.dirichlet_dofs,
                                  task_o.forces, task_o.neumann_nodes, None, task_o.E0,
                                  task_o.nu)


def _fem(task, precision, rtol, pc="auto"):
    from sktopt_amd import fea
    cfg = fea.LinearSolverConfig(rtol=rtol, precision=precision, maxiter=200000,
                                 preconditioner=pc)
    return fea.FEM_SimpLinearElasticity(task, 1e-9, solver_config=cfg)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tet_mg_solve_matches_direct(gpu, precision):
    """24x12x12 jittered tets at a SIMP contrast of ~5e8: the multigrid-
    preconditioned solve equals SuperLU, and in float64 on a random 0/1
    density pattern it needs far fewer iterations than Jacobi-PCG."""
    import torch
    to = oprob.cantilever(24, 12, 12, kind="tet4", jitter=0.2, seed=7)
    rng = np.random.default_rng(0)
    if precision == "fp64":
        # a random 0/1 pattern (moduli 1 and ~2e-9)
        rho = np.where(rng.uniform(size=to.n_elements) < 0.4, 1.0, 1e-3)
    else:
        # the float32 V-cycle breaks down on the random 0/1 pattern; a
        # spatially smooth field spanning the same moduli range converges
        c = to.centers
        rho = np.clip(0.5 + 0.6 * np.sin(c[0] / 3.0) * np.cos(c[2] / 2.0), 1e-3, 1.0)
    E = tr.simp_interpolation(rho, 1.0, 1e-9, 3.0)
    K = to.element_operator().assemble(E)
    F = to.forces[0].copy()
    F[to.dirichlet_dofs] = 0.0
    Ke, _ = ofem.enforce(K, F, to.dirichlet_dofs)
    U_ref = ofem.solve(Ke, F, "spsolve")
    C_ref = float(F @ U_ref)
    res = {}
    # float32 Jacobi-PCG is not claimed at this contrast: the comparison
    # with Jacobi runs in float64
    for pc in (("mg", "jacobi") if precision == "fp64" else ("mg",)):
        fem = _fem(_tet_task(to), precision, 1e-10, pc)
        U = torch.zeros((fem.ndof, 1), dtype=torch.float64, device="cuda")
        C = float(fem.objectives_multi_load(torch.tensor(rho, device="cuda"), 3.0, U)[0])
        res[pc] = (C, fem.last_solve["iters"], fem.last_solve["preconditioner"],
                   fem.last_solve["levels"])
        assert abs(C - C_ref) <= 1e-7 * abs(C_ref), (pc, C, C_ref)
        err = np.abs(U.cpu().numpy()[:, 0] - U_ref).max() / np.abs(U_ref).max()
        assert err <= 1e-6, (pc, err)
    assert res["mg"][2] == "mg" and res["mg"][3] >= 2, res
    print(f"[tet mg {precision}] iterations: {res}", flush=True)
    if precision == "fp64":
        assert res["jacobi"][2] == "jacobi"
        assert res["mg"][1] * 5 < res["jacobi"][1], res


def test_tet_mg_oc_trajectory_matches_oracle(gpu, tmp_path):
    """OC on a 24x12x12 jittered tet cantilever with the multigrid solve,
    float64 at rtol 1e-12, 4 iterations against the oracle's SuperLU loop."""
    from sktopt_amd import core
    from sktopt_amd.tools import SchedulerConfig as SC
    mk = lambda: oprob.cantilever(24, 12, 12, kind="tet4", jitter=0.2, seed=7)  # noqa: E731
    S = odrv.Sched
    ocfg = odrv.Config(max_iters=10, p=S("Constant", 3.0, 3.0), vol_frac=S("Constant", 0.3, 0.3),
                       beta=S("Constant", 1.0, 1.0), filter_radius=S("Constant", 1.5, 1.5),
                       move_limit=S("Constant", 0.2, 0.2), E_min_coeff=1e-9, solver="spsolve")
    loop = odrv.DensityLoop(ocfg, mk())
    cfg = core.OC_Config(dst_path=str(tmp_path), max_iters=10, p=SC.constant(target_value=3.0),
                         vol_frac=SC.constant(target_value=0.3),
                         beta=SC.constant(target_value=1.0), filter_type="spacial",
                         filter_radius=SC.constant(target_value=1.5),
                         move_limit=SC.constant(target_value=0.2), E_min_coeff=1e-9,
                         precision="fp64", solver_rtol=1e-12)
    opt = core.OC_Optimizer(cfg, _tet_task(mk()))
    opt.parameterize()
    for it in range(1, 5):
        rec = loop.step(it)
        opt.optimize_steps(1)
        assert opt.fem.last_solve["preconditioner"] == "mg"
        c = opt.recorder.latest("compliance")
        assert abs(c - rec["compliance"]) <= 1e-9 * abs(rec["compliance"]), (it, c, rec)
        assert opt.recorder.latest("bisection_evals") == rec["n_evals"]
        assert np.abs(opt.rho_host() - loop.rho).max() <= 1e-8, it


def test_tet_100x50x50_oc_iterations(gpu, tmp_path):
    """The tet configuration at size: 100x50x50 cells x 6 jittered tets
    (1.5M tets, 788,103 DOF), r = 1.5 filter, Emin = 1e-9, SIMP p = 3, three
    OC iterations in mixed precision with the multigrid solve.  Checks: the
    true float64 residual of each returned solution, sum_e U_e = C / 2, the
    volume constraint, and the first iteration's compliance against a
    float64 solve of the same state."""
    import time
    import torch
    from sktopt_amd import core
    from sktopt_amd.mesh import toy_problem
    from sktopt_amd.tools import SchedulerConfig as SC
    task = toy_problem.cantilever(100, 50, 50, kind="tet4", jitter=0.2, seed=0)
    assert task.mesh.cell_grid == (100, 50, 50)
    cfg = core.OC_Config(dst_path=str(tmp_path), max_iters=10, p=SC.constant(target_value=3.0),
                         vol_frac=SC.constant(target_value=0.3),
                         beta=SC.constant(target_value=1.0), filter_type="spacial",
                         filter_radius=SC.constant(target_value=1.5),
                         move_limit=SC.constant(target_value=0.2), E_min_coeff=1e-9,
                         precision="mixed", solver_rtol=1e-8)
    opt = core.OC_Optimizer(cfg, task)
    opt.parameterize()
    times = []
    for it in range(3):
        t0 = time.perf_counter()
        opt.optimize_steps(1)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
        ls = opt.fem.last_solve
        assert ls["preconditioner"] == "mg" and ls["converged"], ls
        fem = opt.fem
        U = opt.state["u_dofs"]
        KU = fem.apply(U, E=fem.E64)
        rel = float(torch.linalg.vector_norm(fem.F - KU) / torch.linalg.vector_norm(fem.F))
        assert rel <= 1.05e-8, (it, rel)
        en = float(opt.state["energy"].sum())
        c = opt.recorder.latest("compliance")
        np.testing.assert_allclose(en, 0.5 * c, rtol=1e-7)
        assert abs(opt.recorder.latest("vol_error")) < 1e-4 or \
            opt.recorder.latest("bisection_evals") == 41
        print(f"[tet 100x50x50] it {it + 1}: C={c:.6e} solve iters={ls['iters']} "
              f"levels={ls['levels']} time={times[-1]:.2f}s", flush=True)
    cs = opt.recorder.as_object().compliance
    assert cs[1] < cs[0] and cs[2] < cs[1]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tet_mg_factor2_restriction_matches_row_grid_kernels(gpu, precision, monkeypatch):
    """The tet fine level's residual (zero at Dirichlet DOFs) is restricted
    onto the grid hierarchy by the fused factor-2 kernels (a gather, or tiles
    with SKT_MG_TRANSFERS=tiled), which sum in the order of the two row-grid
    passes (=rowgrid): the solves agree bit for bit."""
    import torch
    from sktopt_amd import fea
    to = oprob.cantilever(16, 8, 8, kind="tet4", jitter=0.2, seed=7)
    c = to.centers
    rho = np.clip(0.5 + 0.6 * np.sin(c[0] / 3.0) * np.cos(c[2] / 2.0), 1e-3, 1.0)
    out = {}
    for mode in ("fused", "tiled", "rowgrid"):
        monkeypatch.setenv("SKT_MG_TRANSFERS", mode)
        cfg = fea.LinearSolverConfig(rtol=1e-10, precision=precision, maxiter=200000,
                                     preconditioner="mg", mg_max_coarse=100)
        fem = fea.FEM_SimpLinearElasticity(_tet_task(to), 1e-9, solver_config=cfg)
        U = torch.zeros((fem.ndof, 1), dtype=torch.float64, device="cuda")
        fem.objectives_multi_load(torch.tensor(rho, device="cuda"), 3.0, U)
        assert fem.last_solve["levels"] >= 3
        out[mode] = (U.cpu().numpy(), fem.last_solve["iters"])
    for mode in ("fused", "tiled"):
        assert out[mode][1] == out["rowgrid"][1]
        np.testing.assert_array_equal(out[mode][0], out["rowgrid"][0])
