"""The bisection makes the decisions at multipliers whose rates are all at
rate_min from one evaluation.  Against the oracle, which evaluates each:
evaluation count, multiplier and densities, for brackets that leave saturation,
that stay in it to the end or never reach it, and where nothing is skipped."""
import numpy as np
import pytest

from oracle import filter as ofilt
from oracle import oc as ooc
from oracle import problems as oprob

pytestmark = pytest.mark.gpu

CASES = {
    # vol_frac, eta, rate_min, l1, l2, tolerance, max_iter, dC
    "usual": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "usual"),
    "volume-too-large-throughout": (0.01, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "usual"),
    "volume-too-small-throughout": (0.99, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "usual"),
    "bracket-below-saturation": (0.3, 0.5, 0.7, 1e-7, 1.5, 1e-5, 1000, "usual"),
    "eta-one": (0.3, 1.0, 0.9, 1e-7, 1e7, 1e-5, 1000, "usual"),
    "eta-two": (0.35, 2.0, 0.5, 1e-7, 1e5, 1e-6, 1000, "usual"),
    "no-lower-rate": (0.3, 0.5, 0.0, 1e-7, 1e7, 1e-5, 1000, "usual"),
    "stopped-by-count": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 5, "usual"),
    "stopped-after-saturation": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 30, "usual"),
    "zero-sensitivities": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "zero"),
    "some-of-the-wrong-sign": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "sign"),
    "not-a-number": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "nan"),
    "infinite": (0.3, 0.5, 0.7, 1e-7, 1e7, 1e-5, 1000, "inf"),
}


@pytest.mark.parametrize("form", ["stencil", "tree", "csr"])
@pytest.mark.parametrize("name", CASES)
def test_matches_oracle(gpu, name, form, monkeypatch):
    import torch
    from sktopt_amd import _lib, mesh as pmesh
    from sktopt_amd.filters import SpacialFilter
    vf, eta, rmin, l1, l2, tol, most, which = CASES[name]
    task = oprob.cantilever(12, 6, 6)
    mask = task.design_mask.copy()
    mask[task.dirichlet_elements] = False
    design = np.nonzero(mask)[0]
    rng = np.random.default_rng(3)
    rho = np.ones(task.n_elements)
    rho[design] = rng.uniform(0.05, 0.9, design.size)
    dC = -rng.uniform(0.0, 1.0, design.size) ** 3
    if which == "zero":
        dC[:] = 0.0
    elif which == "sign":
        dC[::50] *= -1.0
    elif which == "nan":
        dC[7] = np.nan
    elif which == "inf":
        dC[7] = -np.inf
    vol = task.elements_volume[design]
    of = ofilt.SpacialFilter(task.centers, 1.5, mask)
    ref = ooc.bisection_with_physical_volume(
        dC, rho[design], rho, design, of, 1e-2, 1.0, 0.2, eta, 1e-12, vf, 2.0, 0.5, vol,
        vol.sum(), rmin, 1.3, max_iter=most, tolerance=tol, l1=l1, l2=l2)
    monkeypatch.setenv("SKT_OC_TREE", "0" if form == "csr" else "1")
    if form == "stencil":
        f = SpacialFilter(pmesh.structured_hex(12, 6, 6), task.elements_volume, 1.5, mask)
    else:
        f = SpacialFilter(None, task.elements_volume, 1.5, mask, element_centers=task.centers)
    f.handle
    assert f.stencil_active == (form == "stencil")
    t = lambda v: torch.as_tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    a = [t(rho), t(rho[design]), t(dC), t(vol)]
    out = torch.empty(design.size, dtype=torch.float64, device="cuda")
    res = torch.empty(4, dtype=torch.float64, device="cuda")
    for _ in range(2):  # the second call starts from the first one's workspaces
        _lib.call("skt_oc_bisect", f.handle, *[x.data_ptr() for x in a], float(vol.sum()), vf, 0.2,
                  eta, 1e-2, 1.0, rmin, 1.3, 2.0, 0.5, l1, l2, tol, 1e-4, most, out.data_ptr(),
                  res.data_ptr(), torch.cuda.current_stream().cuda_stream)
        r = res.cpu().numpy()
        assert int(r[2]) == ref[3]
        np.testing.assert_allclose(r[0], ref[0], rtol=1e-12)
        # sums of a few hundred terms in another order
        np.testing.assert_allclose(out.cpu().numpy(), ref[2], rtol=1e-12, atol=1e-14)


def test_helmholtz_filter_with_a_small_exponent(gpu, tmp_path):
    """rate_min^(-1 / eta) beyond float64: no multiplier saturates the rates,
    and the design iteration runs as with any other exponent."""
    from sktopt_amd import core
    from sktopt_amd.mesh import toy_problem
    from sktopt_amd.tools import SchedulerConfig as SC
    const = lambda v: SC.constant(target_value=v)  # noqa: E731
    cfg = core.OC_Config(dst_path=str(tmp_path), max_iters=5, p=const(3.0), beta=const(1.0),
                         move_limit=const(0.2), vol_frac=const(0.4), filter_radius=const(1.5),
                         filter_type="helmholtz", eta=const(1e-3), scaling_rate_min=0.1)
    opt = core.OC_Optimizer(cfg, toy_problem.multiload(10, 6, 6, n_loads=1, seed=1))
    opt.parameterize()
    opt.optimize_steps(1)
    assert np.isfinite(opt.rho_host()).all()


@pytest.mark.parametrize("form", ["stencil", "tree", "csr"])
def test_bracket_that_stalls_in_saturation(gpu, form, monkeypatch):
    """A tolerance below the spacing of doubles at the bracket, whose midpoint
    rounds to its lower end: the evaluations end at their bound, ceil(log2(
    width / tolerance)) + 3, also where one serves them all."""
    import torch
    from sktopt_amd import _lib, mesh as pmesh
    from sktopt_amd.filters import SpacialFilter
    m = pmesh.structured_hex(6, 4, 4)
    n = m.nelements
    monkeypatch.setenv("SKT_OC_TREE", "0" if form == "csr" else "1")
    f = SpacialFilter(m, np.ones(n), 1.5)
    f.use_stencil = form == "stencil"
    f.handle
    l1, l2, tol = 1e-7, float(np.nextafter(1e7, np.inf)), 1e-12
    rng = np.random.default_rng(3)
    t = lambda v: torch.as_tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    rho, dC, vol = t(rng.uniform(0.05, 0.9, n)), t(-rng.uniform(0.0, 1.0, n)), t(np.ones(n))
    out, res = torch.empty_like(rho), t(np.zeros(4))
    _lib.call("skt_oc_bisect", f.handle, rho.data_ptr(), rho.data_ptr(), dC.data_ptr(),
              vol.data_ptr(), float(n), 0.01, 0.2, 0.5, 1e-2, 1.0, 0.7, 1.3, 2.0, 0.5, l1, l2, tol,
              1e-4, 1000, out.data_ptr(), res.data_ptr(), torch.cuda.current_stream().cuda_stream)
    r = res.cpu().numpy()
    assert int(r[2]) == int(np.ceil(np.log2((l2 - l1) / tol))) + 3 and r[3] > tol
    expect = np.clip(rho.cpu().numpy() * 0.7, rho.cpu().numpy() - 0.2, rho.cpu().numpy() + 0.2)
    np.testing.assert_allclose(out.cpu().numpy(), np.clip(expect, 1e-2, 1.0), rtol=1e-15)
