"""The structured filter from LDS tiles: forward, adjoint and the bisection's
volume against the CSR form of the same matrix, on grids smaller than a tile,
with remainders along each axis, thin, with holes in the design and with a
radius too wide for the tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [((5, 3, 2), 1.5), ((33, 5, 4), 2.0), ((40, 20, 20), 1.5), ((31, 33, 9), 3.2),
         ((70, 7, 1), 2.0), ((17, 9, 13), 6.5), ((64, 64, 80), 1.2), ((130, 66, 34), 2.0)]


@pytest.mark.parametrize("grid,radius", GRIDS)
@pytest.mark.parametrize("holes", [False, True])
def test_equals_csr(gpu, grid, radius, holes):
    import torch
    from sktopt_amd import _lib, mesh as pmesh
    from sktopt_amd.filters import SpacialFilter
    m = pmesh.structured_hex(*grid)
    rng = np.random.default_rng(1)
    mask = np.ones(m.nelements, dtype=bool)
    if holes:
        mask[rng.choice(m.nelements, m.nelements // 5, replace=False)] = False
    vol = m.elements_volume()
    f, c = (SpacialFilter(m, vol, radius, mask) for _ in range(2))
    c.use_stencil = False
    f.handle, c.handle
    assert f.stencil_active and not c.stencil_active
    x = rng.uniform(size=m.nelements)
    if holes:
        x[np.nonzero(~mask)[0][::3]] = np.nan      # never read into a design row
    x = torch.as_tensor(x, device="cuda")
    for name in ("forward", "gradient"):
        a, b = (getattr(o, name)(x).cpu().numpy() for o in (f, c))
        # up to 250 terms of one sign, summed in another order
        np.testing.assert_allclose(a[mask], b[mask], rtol=1e-14)
        np.testing.assert_array_equal(a[~mask], b[~mask])
    nd = int(mask.sum())
    t = lambda v: torch.as_tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    rho_e, dC, ve = t(rng.uniform(0.05, 0.9, nd)), t(-rng.uniform(size=nd) ** 3), t(vol[mask])
    out = {}
    for o in (f, c):
        r, res = torch.empty_like(rho_e), torch.empty(4, dtype=torch.float64, device="cuda")
        _lib.call("skt_oc_bisect", o.handle, x.data_ptr(), rho_e.data_ptr(), dC.data_ptr(),
                  ve.data_ptr(), float(nd), 0.4, 0.2, 0.5, 1e-2, 1.0, 0.7, 1.3, 2.0, 0.5, 1e-7,
                  1e7, 1e-5, 1e-4, 1000, r.data_ptr(), res.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
        out[o] = r.cpu().numpy(), res.cpu().numpy()
    assert out[f][1][2] == out[c][1][2]
    np.testing.assert_allclose(out[f][1][0], out[c][1][0], rtol=1e-14)
    np.testing.assert_allclose(out[f][1][1], out[c][1][1], atol=1e-12)
    np.testing.assert_array_equal(out[f][0], out[c][0])
