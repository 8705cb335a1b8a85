"""Structured apply on grids small enough that a workgroup takes a few node
planes or a single one: heights around the chunk lengths (a last chunk shorter
than the others, one plane per chunk, one chunk in all), against the assembled
matrix, and the fused dot products over those chunks through a solve."""
import numpy as np
import pytest

from oracle import fem as ofem
from oracle import problems as oprob
from test_gpu_multigrid import _fem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(4, 3, 1), (16, 15, 2), (17, 31, 5), (12, 9, 13), (46, 31, 40),
                                  (61, 61, 7)])
@pytest.mark.parametrize("loads", [1, 4])
def test_apply_matches_assembled(gpu, grid, loads):
    import torch
    task = oprob.multiload(*grid, n_loads=loads, seed=1)
    fem = _fem(task, "elastic", "fp64", 1e-10, "jacobi")
    rng = np.random.default_rng(2)
    E = rng.uniform(1e-9, 1.0, task.n_elements)
    Ke, _ = ofem.enforce(task.element_operator().assemble(E), np.zeros(task.ndof),
                         task.dirichlet_dofs)
    X = rng.standard_normal((task.ndof, loads))
    ref = Ke @ X
    for t, tol in ((torch.float64, 1e-12), (torch.float32, 2e-5)):
        Y = fem.apply(torch.as_tensor(X, dtype=t, device="cuda"),
                      torch.as_tensor(E, dtype=t, device="cuda"), dtype=t)
        assert np.abs(Y.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("grid", [(6, 5, 1), (16, 8, 5), (20, 10, 13)])
def test_solve_matches_direct(gpu, grid):
    task = oprob.multiload(*grid, n_loads=4, seed=3)
    rho = np.random.default_rng(4).uniform(0.1, 1.0, task.n_elements)
    Uo = np.zeros((task.ndof, 4))
    ofem.ElasticFEM(task, 1e-9).objectives_multi_load(rho, 3.0, Uo)
    for precision in ("fp64", "mixed"):
        fem = _fem(task, "elastic", precision, 1e-10, "auto")
        U = np.zeros((task.ndof, 4))
        fem.objectives_multi_load(rho, 3.0, U)
        assert np.abs(U - Uo).max() <= 1e-6 * np.abs(Uo).max()
