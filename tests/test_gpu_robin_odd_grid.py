"""Heat conduction with Robin terms on grids that 2, 3 and 5 do not divide.
The multigrid hierarchy leaves those terms out, so the automatic choice keeps
Jacobi there: strong Robin facets take multigrid many more iterations."""
import numpy as np
import pytest

from test_gpu_heat_robin import _oracle_fem, _task, _tet_oracle_fem, _tet_task

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("h", [4e-2, 1e3])
@pytest.mark.parametrize("mesh", ["hex8", "tet4"])
def test_robin_on_odd_grid_matches_oracle(gpu, mesh, h, precision):
    from sktopt_amd import fea
    if mesh == "hex8":
        t = _task(11, 9, 7, h=h)
        ofem = _oracle_fem(t, "compliance")[1]
    else:
        o, t = _tet_task((7, 7, 7), h=h)
        assert t.mesh.cell_grid == (7, 7, 7)
        ofem = _tet_oracle_fem(o, t, "compliance")
    rho = np.random.default_rng(5).uniform(0.1, 1.0, t.mesh.nelements)
    Uo = np.zeros((t.ndof, 1))
    Jo = ofem.objectives_multi_load(rho, 3.0, Uo)
    its = {}
    for pc in ("auto", "jacobi"):
        cfg = fea.LinearSolverConfig(rtol=1e-10, precision=precision, preconditioner=pc,
                                     mg_max_coarse=100, maxiter=4000)
        fem = fea.FEM_SimpLinearHeatConduction(t, 1e-3, solver_config=cfg)
        U = np.zeros((t.ndof, 1))
        J = fem.objectives_multi_load(rho, 3.0, U)
        assert fem.last_solve["preconditioner"] == "jacobi"
        its[pc] = fem.last_solve["iters"]
        # rtol 1e-10 of the load; the stiff facets' condition number (h / k up
        # to 100) times that
        np.testing.assert_allclose(J, Jo, rtol=1e-6)
        np.testing.assert_allclose(U, Uo, rtol=1e-5, atol=1e-6 * np.abs(Uo).max())
    assert its["auto"] == its["jacobi"]
