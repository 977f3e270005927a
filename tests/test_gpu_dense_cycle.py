"""One V-cycle of a hierarchy whose coarse cycle is a dense matrix, through the public
one-cycle solve, against the cycle restated in numpy on the exported levels: blocks of 6
(SC 16^3: the smallest lattice with three levels, and 20^3) and of 3 (hexagonal)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from lpm_harness import P, get, push
from test_gpu_amg import diag_block_inverses, export, fine_tangent, lambda_max

pytestmark = pytest.mark.gpu


def constrained(case):
    L = P.lib()
    if case == "hex":
        n, x, t, _ = P.build_hex_model([0.0, 90.0, 0.0, 80.0, 0.0, 1.0], critical=1.0)
        P.check(L.lpmx_tangent(), "tangent")
        d = 2
    else:
        n, x, t, _ = P.build_sc_model(P.sc_box_for(case))
        P.check(L.lpmx_tangent(), "tangent")
        d = 3
    dbc = np.ones((n, d), np.int32)
    dbc[t == 2] = 0
    dbc[t == 1, d - 1] = 0
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    return n, d, dbc


def block_diag_apply(Dinv, r, d):
    return np.einsum("iab,ib->ia", Dinv, r.reshape(-1, d)).ravel()


@pytest.mark.parametrize("case", [16, 20, "hex"])
@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_one_cycle(case, prec):
    L = P.lib()
    n, d, dbc = constrained(case)
    b = np.random.default_rng(1).standard_normal(n * d) * dbc.ravel()
    push("RESIDUAL", b)
    P.check(L.lpmx_bc_eliminate(), "eliminate")
    P.check(L.lpmx_set_preconditioner(2), "one cycle")
    it, rr, st = C.c_int(), C.c_double(), C.c_int()
    L.lpmx_solve_ex.argtypes = [C.c_int, C.c_double, C.c_double, C.c_int, C.c_double, C.c_int, C.POINTER(C.c_int),
                                C.POINTER(C.c_double), C.POINTER(C.c_int)]
    P.check(L.lpmx_solve_ex(prec, 1e-8, 0.0, 10, 1e-2, 10, C.byref(it), C.byref(rr), C.byref(st)), "cycle")
    z = get("DISP", (n * d,)).copy()
    lev, ts, by = C.c_int(), C.c_double(), C.c_int64()
    P.check(L.lpmx_amg_info(C.byref(lev), C.byref(ts), C.byref(by)), "info")
    assert lev.value >= 3
    A, levels = fine_tangent(n, d), []
    D = d
    for l in range(lev.value - 1):
        Pl, (_, _, _, bc) = export(l, 1)
        Dinv = diag_block_inverses(A, D)
        hi = 1.15 * lambda_max(A, Dinv, D)
        levels.append((A, Dinv, D, 1.0 / (0.5 * (hi + hi / 10.0)), Pl))
        A, D = (Pl.T @ A @ Pl).tocsr(), bc
    # zero modes of an aggregate: identity, as the device's inverse
    dense = A.toarray()
    zero = np.abs(dense).sum(axis=1) == 0
    dense[zero, zero] = 1.0

    def cycle(l, f):
        if l == len(levels):
            return np.linalg.solve(dense, f)
        Al, Dinv, dl, c, Pl = levels[l]
        x = c * block_diag_apply(Dinv, f, dl)
        x = x + Pl @ cycle(l + 1, Pl.T @ (f - Al @ x))
        return x + c * block_diag_apply(Dinv, f - Al @ x, dl)

    ref = cycle(0, b)
    err = np.abs(z - ref).max() / np.abs(ref).max()
    print(f"{case}: {lev.value} levels, one cycle off by {err:.2e}", flush=True)
    # FP64: rounding through the levels, times the condition (about 1e4) of the coarsest;
    # FP32: its unit, 6e-8, times the same growth over a smoothed residual (measured 1e-6)
    assert err <= (1e-10 if prec == P.LPMX_FP64 else 1e-4)
    P.check(L.lpmx_set_preconditioner(0), "default")
