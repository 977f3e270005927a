"""Block-Jacobi CG on either side of its size rules: p.q summed by every work-group of the
update (up to 1,024 slices) or by a launch of its own, the product from the stored tangent
or over the bonds (from 20,000 particles).  The solution's true residual, formed with the
stored FP64 matrix, against the tolerance asked for."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, push

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge", [8, 24, 28, 40, 41])  # 8, 216, 343, 1,000 and 1,077 slices
@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_true_residual(edge, prec):
    L = P.lib()
    n, x, t, _ = P.build_sc_model(P.sc_box_for(edge))
    P.check(L.lpmx_tangent(), "tangent")
    dbc = np.ones((n, 3), np.int32)
    dbc[t == 2] = 0
    dbc[t == 1, 2] = 0
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    b = np.random.default_rng(edge).standard_normal(3 * n) * dbc.ravel()
    push("RESIDUAL", b)
    P.check(L.lpmx_bc_eliminate(), "eliminate")
    P.check(L.lpmx_set_preconditioner(0), "block-Jacobi")
    it, rr = C.c_int(), C.c_double()
    rtol = 1e-8
    P.check(L.lpmx_solve(prec, rtol * rtol, 0.0, 20000, C.byref(it), C.byref(rr)), "solve")
    z, y = np.ascontiguousarray(get("DISP", (3 * n,))), np.zeros(3 * n)
    P.check(L.lpmx_spmv(P.LPMX_FP64, P.ptr(z), P.ptr(y)), "product")
    # FP64: the recurrence's residual drifts from the true one by about its unit, 1.1e-16,
    # times the condition (about edge^2) and the iterations, far below; mixed: true residual
    assert np.linalg.norm(b - y) <= 1.01 * rtol * np.linalg.norm(b)
    assert it.value > 5
