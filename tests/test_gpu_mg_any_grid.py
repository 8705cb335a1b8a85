"""Multigrid on grids of any size: levels are halved on every axis, and the
last coarse element of an odd axis holds one fine element.  Solutions against
the oracle's direct solve, the fused restriction against the two-pass one, and
the routes such grids took before that stay as they were."""
import numpy as np
import pytest

from oracle import fem as ofem
from oracle import problems as oprob
from test_gpu_multigrid import _fem

pytestmark = pytest.mark.gpu

GRIDS = [
    # name, task factory, physics, max_coarse
    ("odd-on-every-axis", lambda: oprob.multiload(13, 11, 9, n_loads=3, seed=1), "elastic", 100),
    ("odd-below-the-fine-level", lambda: oprob.multiload(22, 10, 14, n_loads=2, seed=2), "elastic",
     60),
    ("one-element-thick", lambda: oprob.multiload(41, 23, 1, n_loads=1, seed=3), "elastic", 60),
    ("two-elements-thick", lambda: oprob.multiload(29, 2, 31, n_loads=4, seed=4), "elastic", 200),
    ("prime-heat", lambda: oprob.heat_patch(17, patch=4), "heat", 30),
]


def _densities(task):
    return np.random.default_rng(6).uniform(0.02, 1.0, task.n_elements)


@pytest.mark.parametrize("precision,rtol,ctol", [("fp64", 1e-12, 1e-9), ("mixed", 1e-10, 1e-8)])
@pytest.mark.parametrize("name,mk,physics,max_coarse", GRIDS)
def test_solve_matches_direct(gpu, precision, rtol, ctol, name, mk, physics, max_coarse,
                              monkeypatch):
    task = mk()
    rho = _densities(task)
    ofe = ofem.ElasticFEM(task, 1e-9) if physics == "elastic" else ofem.HeatFEM(task, 1e-3)
    Uo = np.zeros((task.ndof, task.n_tasks))
    co = ofe.objectives_multi_load(rho, 3.0, Uo)
    out, its = {}, {}
    for mode in ("fused", "tiled", "rowgrid"):
        monkeypatch.setenv("SKT_MG_TRANSFERS", mode)
        fem = _fem(task, physics, precision, rtol, "auto", max_coarse)
        U = np.zeros((task.ndof, task.n_tasks))
        c = fem.objectives_multi_load(rho, 3.0, U)
        assert fem.last_solve["preconditioner"] == "mg" and fem.last_solve["levels"] >= 3
        np.testing.assert_allclose(c, co, rtol=ctol)
        assert np.abs(U - Uo).max() <= 1e-6 * np.abs(Uo).max()
        out[mode], its[mode] = U, fem.last_solve["iters"]
    # the same sums in the same order
    for mode in ("fused", "tiled"):
        assert its[mode] == its["rowgrid"]
        np.testing.assert_array_equal(out[mode], out["rowgrid"])
    fem = _fem(task, physics, precision, rtol, "jacobi", max_coarse)
    fem.objectives_multi_load(rho, 3.0, np.zeros((task.ndof, task.n_tasks)))
    print(f"[{name} {precision}] iterations {its['fused']}, Jacobi {fem.last_solve['iters']}")
    assert 2 * its["fused"] <= fem.last_solve["iters"]


@pytest.mark.parametrize("grid,precision", [((65, 17, 503), "mixed"), ((65, 17, 251), "fp64"),
                                            ((64, 17, 252), "mixed"), ((63, 31, 64), "fp64")])
def test_tiled_restriction_of_large_levels(gpu, grid, precision, monkeypatch):
    """Levels that take the tiled factor-2 kernel, with 8 columns, in chunks of
    4, 2, 2 and 1 coarse planes; on the first three the last coarse plane is
    alone in its chunk, at an odd end of the axis or not.  Two iterations, bit
    for bit those of the row-grid kernels."""
    from dataclasses import replace
    nx, ny, nz = grid
    node = np.arange((nx + 1) * (ny + 1) * (nz + 1)).reshape(nz + 1, ny + 1, nx + 1)
    task = oprob.multiload(4, 4, 4, n_loads=8, seed=1)
    from oracle import mesh as om
    task.mesh = om.structured_hex(*grid)
    task.dirichlet_nodes = node[0].ravel()
    task.dirichlet_dofs = (3 * node[0].ravel()[:, None] + np.arange(3)).ravel()
    f = np.zeros((8, node.size * 3))
    f[np.arange(8), 3 * node[-1, :, -1][:8] + np.arange(8) % 3] = 1.0
    f[:, ::7] += 1e-3 * np.random.default_rng(2).standard_normal(f[:, ::7].shape)
    f[:, task.dirichlet_dofs] = 0.0
    task.forces = list(f)
    rho = np.random.default_rng(6).uniform(0.02, 1.0, nx * ny * nz)
    out = {}
    for mode in ("tiled", "rowgrid"):
        monkeypatch.setenv("SKT_MG_TRANSFERS", mode)
        fem = _fem(task, "elastic", precision, 1e-10, "auto")
        fem.solver_config = replace(fem.solver_config, maxiter=2, on_noconv="warn")
        out[mode] = np.zeros((node.size * 3, 8))
        fem.objectives_multi_load(rho, 3.0, out[mode])
        assert fem.last_solve["preconditioner"] == "mg" and fem.last_solve["iters"] == 2
    assert np.abs(out["tiled"]).max() > 0
    np.testing.assert_array_equal(out["tiled"], out["rowgrid"])


def test_tet_grid_of_odd_cells_matches_jacobi(gpu):
    from sktopt_amd import fea
    from sktopt_amd.mesh import toy_problem
    task = toy_problem.cantilever(13, 7, 9, kind="tet4", jitter=0.2, seed=2)
    rho = np.random.default_rng(7).uniform(0.05, 1.0, task.mesh.nelements)
    out = {}
    for pc in ("auto", "jacobi"):
        cfg = fea.LinearSolverConfig(rtol=1e-12, precision="fp64", preconditioner=pc,
                                     mg_max_coarse=100)
        fem = fea.FEM_SimpLinearElasticity(task, 1e-6, solver_config=cfg)
        U = np.zeros((fem.ndof, 1))
        fem.objectives_multi_load(rho, 3.0, U)
        out[pc] = U
        assert fem.last_solve["preconditioner"] == ("mg" if pc == "auto" else "jacobi")
    assert np.abs(out["auto"] - out["jacobi"]).max() <= 1e-8 * np.abs(out["jacobi"]).max()


@pytest.mark.parametrize("cells", [(7, 7, 7), (8, 8, 8)])
@pytest.mark.parametrize("columns", [1, 2, 3, 4, 5])
def test_tet_heat_of_any_number_of_columns(gpu, cells, columns):
    """Tet operators take all columns as one block; the cycle is built for
    blocks of 1, 2 and 4 scalar columns, the others are Jacobi's."""
    from sktopt_amd import fea, mesh as pmesh
    m = pmesh.jittered_tet(*cells, jitter=0.2, seed=3)
    n = (cells[0] + 1) * (cells[1] + 1)
    values = [100.0 * (c + 1) for c in range(columns)]
    t = pmesh.LinearHeatConduction(m, np.arange(n), values, np.ones(m.nvertices), None, 1.0)
    rho = np.random.default_rng(7).uniform(0.05, 1.0, m.nelements)
    out = {}
    for pc in ("auto", "jacobi"):
        cfg = fea.LinearSolverConfig(rtol=1e-12, precision="fp64", preconditioner=pc,
                                     mg_max_coarse=100)
        fem = fea.FEM_SimpLinearHeatConduction(t, 1e-3, solver_config=cfg)
        out[pc] = np.zeros((m.nvertices, columns))
        fem.objectives_multi_load(rho, 3.0, out[pc])
        mg = pc == "auto" and columns in (1, 2, 4)
        assert fem.last_solve["preconditioner"] == ("mg" if mg else "jacobi")
    assert np.abs(out["auto"] - out["jacobi"]).max() <= 1e-8 * np.abs(out["jacobi"]).max()


def test_explicit_request_stays_refused(gpu):
    """Factors 2, 3 and 5 do not reach 100 DOFs from 13 x 11 x 7 elements."""
    task = oprob.cantilever(13, 11, 7)
    fem = _fem(task, "elastic", "fp64", 1e-8, "mg", 100)
    with pytest.raises(ValueError, match="factors 2, 3 and 5 divide"):
        fem.objectives_multi_load(_densities(task), 3.0, np.zeros((task.ndof, 1)))


@pytest.mark.parametrize("keep", [0, 1])
def test_mass_operator_takes_it_where_one_set_up_serves_all_solves(gpu, keep):
    """A Helmholtz operator on a grid that 2, 3 and 5 do not divide: Jacobi with
    a set-up per solve, multigrid with one for all (as the filter asks for)."""
    import ctypes as C
    import torch
    from sktopt_amd import _lib
    n, e = 24 * 20 * 14, 23 * 19 * 13
    t = dict(dtype=torch.float64, device="cuda")
    fixed, E, F = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.ones(e, **t), \
        torch.rand((n, 1), **t)
    op, s = C.c_void_p(), C.c_void_p()
    _lib.call("skt_hex8_create_scalar", 23, 19, 13, 1.0, 1.0, 1.0, 1.0, 4.0, fixed.data_ptr(),
              C.byref(op))
    _lib.call("skt_solver_create", op, 1, C.byref(s))
    _lib.call("skt_solver_fix_moduli", s, keep)
    U, it, rr = torch.zeros((n, 1), **t), (C.c_int64 * 2)(), (C.c_double * 1)()
    _lib.call("skt_solver_solve", s, _lib.F64, 1, E.data_ptr(), None, F.data_ptr(), U.data_ptr(),
              1e-10, 1000, 0.0, it, rr, torch.cuda.current_stream().cuda_stream)
    pc, lev = C.c_int(), C.c_int()
    _lib.call("skt_solver_info", s, C.byref(pc), C.byref(lev))
    assert pc.value == (_lib.PC_MG if keep else _lib.PC_JACOBI) and rr[0] <= 1e-10
    _lib.load().skt_solver_destroy(s)
    _lib.load().skt_operator_destroy(op)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", [(13, 11, 9), (16, 12, 8)])
def test_a_cycle_that_breaks_down_falls_back_to_jacobi(gpu, grid, precision, monkeypatch):
    """SKT_MG_MARGIN = 0.4 smooths with less than half of the largest
    eigenvalue, so the cycle is not definite: the solve is Jacobi's, with the
    multigrid iterations counted; after two of them Jacobi alone; a solver that
    is configured anew tries multigrid again."""
    from sktopt_amd import _lib
    task = oprob.multiload(*grid, n_loads=2, seed=1)
    rho = np.where(np.random.default_rng(3).uniform(size=task.n_elements) < 0.5, 1.0, 1e-3)
    Uo = np.zeros((task.ndof, 2))
    co = ofem.ElasticFEM(task, 1e-9).objectives_multi_load(rho, 3.0, Uo)
    ref = _fem(task, "elastic", precision, 1e-10, "jacobi", 100)
    ref.objectives_multi_load(rho, 3.0, np.zeros((task.ndof, 2)))
    alone = ref.last_solve["iters"]
    monkeypatch.setenv("SKT_MG_MARGIN", "0.4")
    fem = _fem(task, "elastic", precision, 1e-10, "auto", 100)

    def solve():
        U = np.zeros((task.ndof, 2))
        np.testing.assert_allclose(fem.objectives_multi_load(rho, 3.0, U), co, rtol=1e-7)
        return fem.last_solve
    for extra in (True, True, False, False):
        last = solve()
        assert last["preconditioner"] == "jacobi"
        assert (last["iters"] > alone) if extra else (last["iters"] == alone)
    _lib.call("skt_solver_configure", fem._solver, _lib.PC_AUTO, 2, 100)
    assert solve()["iters"] > alone
    monkeypatch.delenv("SKT_MG_MARGIN")
    fem = _fem(task, "elastic", precision, 1e-10, "auto", 100)
    assert solve()["preconditioner"] == "mg"


def test_slightly_indefinite_cycle_keeps_multigrid(gpu, monkeypatch):
    """With 0.9 of the largest eigenvalue r.z is negative now and then, but the
    solve converges, in a fifth of Jacobi's iterations."""
    monkeypatch.setenv("SKT_MG_MARGIN", "0.9")
    task = oprob.multiload(13, 11, 9, n_loads=2, seed=1)
    rho = np.where(np.random.default_rng(3).uniform(size=task.n_elements) < 0.5, 1.0, 1e-3)
    co = ofem.ElasticFEM(task, 1e-9).objectives_multi_load(rho, 3.0, np.zeros((task.ndof, 2)))
    fem = _fem(task, "elastic", "fp64", 1e-10, "auto", 100)
    c = fem.objectives_multi_load(rho, 3.0, np.zeros((task.ndof, 2)))
    np.testing.assert_allclose(c, co, rtol=1e-7)
    assert fem.last_solve["preconditioner"] == "mg" and 80 < fem.last_solve["iters"] < 200


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_spent_iterations_are_not_a_breakdown(gpu, precision):
    """A multigrid solve that runs out of iterations ends there."""
    from dataclasses import replace
    task = oprob.multiload(13, 11, 9, n_loads=2, seed=1)
    fem = _fem(task, "elastic", precision, 1e-10, "auto", 100)
    fem.solver_config = replace(fem.solver_config, maxiter=4, on_noconv="warn")
    fem.objectives_multi_load(_densities(task), 3.0, np.zeros((task.ndof, 2)))
    last = fem.last_solve
    assert last["preconditioner"] == "mg" and last["iters"] == 4 and not last["converged"]


@pytest.mark.parametrize("grid", [(32, 16, 16), (96, 34, 34)])
@pytest.mark.parametrize("loads", [6, 8])
def test_column_groups_per_workgroup_give_the_same_bits(gpu, grid, loads, monkeypatch):
    """Coarse stencil applies with one column group per workgroup (few tiles)
    or several (level of 48 x 17 x 17 elements), the last one partly filled:
    bit for bit the node-major kernel's, which takes one group per thread."""
    task = oprob.multiload(*grid, n_loads=loads, seed=7)
    rho = _densities(task)
    out = {}
    for layout in ("node", "small"):
        monkeypatch.setenv("SKT_MG_STENCIL_LAYOUT", layout)
        fem = _fem(task, "elastic", "mixed", 1e-8, "auto")
        U = np.zeros((task.ndof, loads))
        fem.objectives_multi_load(rho, 3.0, U)
        out[layout] = U, fem.last_solve["iters"]
    assert out["node"][1] == out["small"][1]
    np.testing.assert_array_equal(out["node"][0], out["small"][0])


@pytest.mark.parametrize("grid,coarse", [((6, 6, 6), 64), ((4, 6, 8), 60), ((8, 8, 6), 100),
                                         ((10, 6, 8), 120), ((14, 8, 6), 160), ((14, 14, 14), 512),
                                         ((20, 12, 8), 385)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_coarsest_inverse_sizes(gpu, grid, coarse, precision):
    """Two levels whose coarsest matrix has one row less, as many, or a few more
    than a multiple of the pivot block's 64 rows.  With an exact coarse solve the
    cycle contracts fast; a wrong inverse would not converge in these counts."""
    task = oprob.heat_patch(grid[0], patch=3)
    from oracle import mesh as om
    task.mesh = om.structured_hex(*grid)
    task.dirichlet_dofs = np.arange(0, (grid[0] + 1) * (grid[1] + 1), 3)
    task.dirichlet_nodes = task.dirichlet_dofs
    task.forces = [np.ones(task.mesh.nnodes)]
    rho = np.random.default_rng(8).uniform(0.3, 1.0, task.mesh.nelements)
    ofe = ofem.HeatFEM(task, 1e-3)
    Uo = np.zeros((task.mesh.nnodes, 1))
    ofe.objectives_multi_load(rho, 3.0, Uo)
    fem = _fem(task, "heat", precision, 1e-10, "mg", coarse)
    U = np.zeros((task.mesh.nnodes, 1))
    fem.objectives_multi_load(rho, 3.0, U)
    assert fem.last_solve["levels"] == 2 and fem.last_solve["iters"] <= 24
    assert np.abs(U - Uo).max() <= 1e-7 * np.abs(Uo).max()
