"""Restriction into a level coarsened by 3 on an axis: where its rows are few,
the plane sums gather all fine nodes of a coarse one at once.  The same sums in
the same order as the row-grid kernel, so the solves agree bit for bit."""
import numpy as np
import pytest

from oracle import problems as oprob
from test_gpu_multigrid import _fem

pytestmark = pytest.mark.gpu

GRIDS = {
    # task factory, physics, max_coarse, levels; factors of the level taken by 3
    "three-axes": (lambda: oprob.multiload(27, 9, 9, n_loads=2, seed=1), "elastic", 480, 2),  # 3 3 3
    "mixed-ragged": (lambda: oprob.multiload(33, 17, 13, n_loads=3, seed=2), "elastic", 2000,
                     2),                                                               # 3 3 3
    "one-load": (lambda: oprob.multiload(15, 6, 9, n_loads=1, seed=3), "elastic", 300, 2),  # 3 2 3
    "four-loads": (lambda: oprob.multiload(18, 6, 8, n_loads=4, seed=4), "elastic", 300,
                   2),                                                                 # 3 3 3
    "heat": (lambda: oprob.heat_patch(18, patch=4), "heat", 30, 4),                    # 3 3 3
}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", GRIDS)
def test_same_solve_as_row_grid(gpu, name, precision, monkeypatch):
    mk, physics, max_coarse, levels = GRIDS[name]
    task = mk()
    rho = np.random.default_rng(8).uniform(0.05, 1.0, task.n_elements)
    out = {}
    for mode in ("fused", "rowgrid"):
        monkeypatch.setenv("SKT_MG_TRANSFERS", mode)
        fem = _fem(task, physics, precision, 1e-10, "auto", max_coarse=max_coarse)
        U = np.zeros((task.ndof, task.n_tasks))
        fem.objectives_multi_load(rho, 3.0, U)
        assert fem.last_solve["preconditioner"] == "mg"
        assert fem.last_solve["levels"] == levels
        out[mode] = (U, fem.last_solve["iters"])
    assert out["fused"][1] == out["rowgrid"][1]
    np.testing.assert_array_equal(out["fused"][0], out["rowgrid"][0])
