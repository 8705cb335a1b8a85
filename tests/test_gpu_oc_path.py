"""From 2^22 entries of the filter matrix on, a pass of the CSR bisection
evaluates the midpoints on the way to the multiplier that is expected.  One
midpoint at a time takes the same decisions: evaluation count, multiplier,
volume error, bracket and densities bit for bit, also where the expectation
fails (densities at their limits, sensitivities of both signs or NaN)."""
import numpy as np
import pytest

from oracle import problems as oprob

pytestmark = pytest.mark.gpu

CALLS = [  # vol_frac, eta, rate_min, l1, l2, tolerance, vol_tol, max_iter
    (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1e-4, 1000),
    (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-9, 1e-13, 1000),
    (0.45, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1e-6, 1000),
    (0.4, 1.0, 0.9, 1e-7, 1e7, 1e-8, 1e-9, 1000),
    (0.35, 2.0, 0.5, 1e-7, 1e5, 1e-6, 1e-7, 1000),
    (0.3, 0.5, 0.0, 1e-7, 1e7, 1e-5, 1e-8, 1000),
    (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-9, 1e-12, 33),
    (0.3, 0.5, 0.7, 0.01, 1.5, 1e-9, 1e-12, 1000),
    (0.3, 0.5, 0.7, -1.0, 2.0, 1e-6, 1e-9, 1000),
    (0.01, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1e-4, 1000),
    (0.99, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1e-4, 1000),
    (0.4, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1e-4, 0),
]


@pytest.mark.parametrize("which", ["usual", "steep", "sign", "nan"])
def test_same_as_one_midpoint_at_a_time(gpu, which, monkeypatch):
    import torch
    from sktopt_amd import _lib
    from sktopt_amd.filters import SpacialFilter
    task = oprob.cantilever(20, 12, 10)
    mask = task.design_mask.copy()
    mask[task.dirichlet_elements] = False
    design = np.nonzero(mask)[0]
    rng = np.random.default_rng(7)
    rho = np.ones(task.n_elements)
    rho[design] = rng.uniform(0.05, 0.9, design.size)
    dC = -rng.uniform(0.0, 1.0, design.size) ** (40 if which == "steep" else 3)
    if which == "sign":
        dC[::50] *= -1.0
    elif which == "nan":
        dC[7] = np.nan
    vol = task.elements_volume[design]
    f = SpacialFilter(None, task.elements_volume, 26.0, mask, element_centers=task.centers)
    f.handle
    assert f.nnz >= 1 << 22 and not f.stencil_active
    a = [torch.as_tensor(v, dtype=torch.float64, device="cuda")
         for v in (rho, rho[design], dC, vol)]
    s = torch.cuda.current_stream().cuda_stream
    for vf, eta, rmin, l1, l2, tol, vtol, most in CALLS:
        got = {}
        for tree in ("1", "0"):
            monkeypatch.setenv("SKT_OC_TREE", tree)
            o = torch.empty(design.size, dtype=torch.float64, device="cuda")
            r = torch.empty(4, dtype=torch.float64, device="cuda")
            _lib.call("skt_oc_bisect", f.handle, *[x.data_ptr() for x in a], float(vol.sum()), vf,
                      0.2, eta, 1e-2, 1.0, rmin, 1.3, 2.0, 0.5, l1, l2, tol, vtol, most,
                      o.data_ptr(), r.data_ptr(), s)
            got[tree] = (r.cpu().numpy(), o.cpu().numpy())
        what = f"{which}: vf {vf} eta {eta} l1 {l1} most {most}"
        np.testing.assert_array_equal(got["1"][0], got["0"][0], err_msg=what)
        np.testing.assert_array_equal(got["1"][1], got["0"][1], err_msg=what)
