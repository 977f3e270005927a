"""Which form the products take and how many bytes they move is what the next solve does,
whether or not a solve has been run on this tangent (27^3 and 28^3 particles: either side of
the bond form's size rule)."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, push

pytestmark = pytest.mark.gpu


def described(prec):
    L = P.lib()
    a, b, c, ms = C.c_double(), C.c_double(), C.c_double(), C.c_double()
    P.check(L.lpmx_bench_spmv(prec, 2, C.byref(ms), C.byref(c)), "bench")
    P.check(L.lpmx_spmv_bytes(prec, C.byref(a)), "product bytes")
    P.check(L.lpmx_amg_smoother_bytes(prec, C.byref(b)), "smoother bytes")
    assert ms.value > 0 and c.value == a.value
    return a.value, b.value, L.lpmx_bond_form_used()


@pytest.mark.parametrize("edge,bonds", [(27, 0), (28, 1)])
@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_described_before_and_after_a_solve(edge, bonds, prec):
    L = P.lib()
    n, x, t, _ = P.build_sc_model(P.sc_box_for(edge))
    P.check(L.lpmx_tangent(), "tangent")
    whole = described(prec)
    assert whole[2] == 0  # without the constraints there is no bond form
    dbc = np.ones((n, 3), np.int32)
    dbc[t == 2] = 0
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    b = np.random.default_rng(edge).standard_normal(3 * n) * dbc.ravel()
    push("RESIDUAL", b)
    P.check(L.lpmx_bc_eliminate(), "eliminate")
    before = described(prec)
    P.check(L.lpmx_set_preconditioner(0), "block-Jacobi")
    it, rr = C.c_int(), C.c_double()
    P.check(L.lpmx_solve(prec, 1e-8, 0.0, 20000, C.byref(it), C.byref(rr)), "solve")
    assert described(prec) == before and before[2] == bonds
    assert (before[:2] == whole[:2]) == (bonds == 0)
    z, y = np.ascontiguousarray(get("DISP", (3 * n,))), np.zeros(3 * n)
    P.check(L.lpmx_spmv(P.LPMX_FP64, P.ptr(z), P.ptr(y)), "product")
    # the bench's product before the solve leaves nothing behind in it
    assert np.linalg.norm(b - y) <= 1.01e-4 * np.linalg.norm(b)
