"""Solvers told that their moduli stay the same set up once: the later solves
give what a solver that sets up every time gives, in both modes, after a change
of mode and after a change of the preconditioner."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(20, 16, 14), (23, 19, 13)])
def test_later_solves_equal_fresh_set_ups(gpu, grid):
    import torch
    from sktopt_amd import _lib
    n = int(np.prod([g + 1 for g in grid]))
    dev = dict(dtype=torch.float64, device="cuda")
    fixed = torch.zeros(n, dtype=torch.uint8, device="cuda")
    E = torch.ones(int(np.prod(grid)), **dev)
    E32 = E.float()
    op = C.c_void_p()
    _lib.call("skt_hex8_create_scalar", *grid, 1.0, 1.0, 1.0, 1.0, 4.0, fixed.data_ptr(),
              C.byref(op))
    s = {}
    for keep in (0, 1):
        s[keep] = C.c_void_p()
        _lib.call("skt_solver_create", op, 2, C.byref(s[keep]))
        _lib.call("skt_solver_fix_moduli", s[keep], keep)
    gen = torch.Generator(device="cuda").manual_seed(1)
    for step, mode in enumerate((_lib.F64, _lib.F64, _lib.F32, _lib.F32, _lib.F64, _lib.F64)):
        if step == 5:
            for v in s.values():
                _lib.call("skt_solver_configure", v, _lib.PC_JACOBI, 2, 2000)
        F = torch.rand((n, 2), generator=gen, **dev)
        out = {}
        for keep, v in s.items():
            U = torch.zeros((n, 2), **dev)
            it, rr = (C.c_int64 * 2)(), (C.c_double * 2)()
            _lib.call("skt_solver_solve", v, mode, 2, E.data_ptr(), E32.data_ptr(), F.data_ptr(),
                      U.data_ptr(), 1e-11, 5000, 0.0, it, rr,
                      torch.cuda.current_stream().cuda_stream)
            assert max(rr) <= 1e-11
            out[keep] = U.cpu().numpy()
        # the power iteration of a repeated set-up refines the smoother's
        # bound, so the iterates differ within the residual's tolerance (the
        # operator's condition number is below 100)
        assert np.abs(out[1] - out[0]).max() <= 2e-9 * np.abs(out[0]).max()
    for v in s.values():
        _lib.load().skt_solver_destroy(v)
    _lib.load().skt_operator_destroy(op)


@pytest.mark.parametrize("order", [(1, 3, 1), (3, 1, 3)])
def test_column_counts_on_a_grid_of_tets(gpu, order):
    """Tets block all columns of a solve, and multigrid is built for one or two
    of elasticity: each solve of the solver takes what its own count allows."""
    import torch
    from sktopt_amd import _lib, fea
    from sktopt_amd.mesh import toy_problem
    t = toy_problem.cantilever(8, 7, 6, kind="tet4", jitter=0.2, seed=2)
    op = fea.FEM_SimpLinearElasticity(t, 1e-6)
    n, dev = op.ndof, dict(dtype=torch.float64, device="cuda")
    E = torch.ones(op.n_el, **dev)
    free = 1.0 - torch.as_tensor(t.dof_fixed_mask(), device="cuda").double()[:, None]
    F = free * torch.rand((n, 3), generator=torch.Generator(device="cuda").manual_seed(1), **dev)
    s = C.c_void_p()
    _lib.call("skt_solver_create", op._op, 3, C.byref(s))
    _lib.call("skt_solver_configure", s, _lib.PC_AUTO, 2, 100)
    _lib.call("skt_solver_fix_moduli", s, 1)
    for k in order:
        U, f = torch.zeros((n, k), **dev), F[:, :k].contiguous()
        it, rr = (C.c_int64 * 2)(), (C.c_double * 3)()
        _lib.call("skt_solver_solve", s, _lib.F64, k, E.data_ptr(), None, f.data_ptr(),
                  U.data_ptr(), 1e-10, 5000, 0.0, it, rr, torch.cuda.current_stream().cuda_stream)
        pc, lev = C.c_int(), C.c_int()
        _lib.call("skt_solver_info", s, C.byref(pc), C.byref(lev))
        assert pc.value == (_lib.PC_MG if k == 1 else _lib.PC_JACOBI) and max(rr[:k]) <= 1e-10
        R = f - op.apply(U, E)
        assert (R * free).norm() <= 1e-9 * f.norm()
    _lib.load().skt_solver_destroy(s)


def test_timing_switched_between_solves(gpu):
    """The V-cycle's timing follows the solver's also where a solve keeps the
    set-up of an earlier one."""
    import torch
    from sktopt_amd import _lib
    g = (20, 16, 14)
    n, dev = 21 * 17 * 15, dict(dtype=torch.float64, device="cuda")
    fixed, E = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.ones(20 * 16 * 14, **dev)
    F, op, s = torch.rand((n, 1), **dev), C.c_void_p(), C.c_void_p()
    _lib.call("skt_hex8_create_scalar", *g, 1.0, 1.0, 1.0, 1.0, 4.0, fixed.data_ptr(), C.byref(op))
    _lib.call("skt_solver_create", op, 1, C.byref(s))
    _lib.call("skt_solver_fix_moduli", s, 1)
    for on in (0, 1, 0):
        _lib.call("skt_solver_set_timing", s, on)
        U, it, rr = torch.zeros((n, 1), **dev), (C.c_int64 * 2)(), (C.c_double * 1)()
        _lib.call("skt_solver_solve", s, _lib.F64, 1, E.data_ptr(), None, F.data_ptr(),
                  U.data_ptr(), 1e-10, 1000, 0.0, it, rr, torch.cuda.current_stream().cuda_stream)
        ms, cnt = (C.c_double * 4)(), (C.c_int64 * 4)()
        _lib.call("skt_solver_get_vcycle_timing", s, ms, cnt, 1)
        assert rr[0] <= 1e-10 and (sum(cnt) > 0) == bool(on)
    _lib.load().skt_solver_destroy(s)
    _lib.load().skt_operator_destroy(op)
