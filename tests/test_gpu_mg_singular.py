"""State solves whose operator is singular: bodies without supports, or on
rollers, under balanced loads, and conduction without Dirichlet nodes.  CG
solves them with any definite preconditioner, so the multigrid has to be one:
on grids that 2, 3 and 5 divide and on others, in both precisions."""
import numpy as np
import pytest

from oracle import mesh as om
from oracle import problems as oprob
from test_gpu_multigrid import _fem

pytestmark = pytest.mark.gpu


def _task(kind, g):
    nx, ny, nz = g
    node = np.arange((nx + 1) * (ny + 1) * (nz + 1)).reshape(nz + 1, ny + 1, nx + 1)
    if kind == "heat":
        t = oprob.heat_patch(nx, patch=2)
        t.mesh = om.structured_hex(*g)
        t.dirichlet_dofs = t.dirichlet_nodes = np.zeros(0, dtype=np.int64)
        q = np.random.default_rng(1).standard_normal(node.size)
        t.forces = [q - q.mean()]
        return t
    t = oprob.multiload(*g, n_loads=1, seed=1)
    f = np.zeros((node.size, 3))
    f[node[:, :, 0], 0], f[node[:, :, -1], 0] = -1.0, 1.0      # tension along x
    t.forces = [f.ravel()]
    d = {"free": np.zeros(0, dtype=np.int64), "rollers": 3 * node[0].ravel() + 2}[kind]
    t.dirichlet_dofs, t.dirichlet_nodes = d, np.unique(d // 3)
    return t


def _solve(t, kind, precision, pc):
    from dataclasses import replace
    fem = _fem(t, "heat" if kind == "heat" else "elastic", precision, 1e-8, pc)
    fem.solver_config = replace(fem.solver_config, maxiter=1000)
    rho = np.random.default_rng(5).uniform(0.1, 1.0, t.n_elements)
    U = np.zeros((t.ndof, 1))
    return fem.objectives_multi_load(rho, 3.0, U), fem.last_solve


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", [(33, 17, 13), (32, 16, 16)])
@pytest.mark.parametrize("kind", ["free", "rollers", "heat"])
def test_multigrid_converges_without_supports(gpu, kind, grid, precision):
    t = _task(kind, grid)
    c, last = _solve(t, kind, precision, "auto")
    assert last["preconditioner"] == "mg" and last["converged"] and last["iters"] <= 60
    # the energy does not see the null space; both solves stop at 1e-8
    np.testing.assert_allclose(c, _solve(t, kind, precision, "jacobi")[0], rtol=1e-6)
    if grid == (32, 16, 16):
        assert _solve(t, kind, precision, "mg")[1]["converged"]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["free", "rollers"])
def test_tet_grid_without_supports(gpu, kind, precision):
    """The same on jittered tets, whose rigid rotations the grid's
    interpolation holds only approximately."""
    from sktopt_amd import fea
    from sktopt_amd.mesh import toy_problem
    t = toy_problem.cantilever(13, 7, 9, kind="tet4", jitter=0.2, seed=2)
    h = _task(kind, (13, 7, 9))
    t.neumann_linear, t.dirichlet_dofs, t.dirichlet_nodes = h.forces, h.dirichlet_dofs, \
        h.dirichlet_nodes
    rho = np.random.default_rng(7).uniform(0.05, 1.0, t.mesh.nelements)
    c = {}
    for pc in ("auto", "jacobi"):
        cfg = fea.LinearSolverConfig(rtol=1e-8, precision=precision, preconditioner=pc,
                                     mg_max_coarse=100, maxiter=1000)
        fem = fea.FEM_SimpLinearElasticity(t, 1e-6, solver_config=cfg)
        U = np.zeros((fem.ndof, 1))
        c[pc] = fem.objectives_multi_load(rho, 3.0, U)
        assert fem.last_solve["preconditioner"] == ("mg" if pc == "auto" else "jacobi")
    np.testing.assert_allclose(c["auto"], c["jacobi"], rtol=1e-6)
