"""With the card full (LPMX_MALLOC_TIGHT) nothing fails for memory that only makes something
faster: the bond form gives way to a hierarchy that needs room, is not made when there is
none, and a level whose dense cycle does not fit keeps its launches."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, push

pytestmark = pytest.mark.gpu


def tangent(n, t):
    L = P.lib()
    P.check(L.lpmx_tangent(), "tangent")
    dbc = np.ones((n, 3), np.int32)
    dbc[t == 2] = 0
    dbc[t == 1, 2] = 0
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    P.check(L.lpmx_bc_eliminate(), "eliminate")
    return dbc.ravel()


def solve(n, b, kind, prec):
    L = P.lib()
    push("RESIDUAL", b)
    P.check(L.lpmx_set_preconditioner(kind), "preconditioner")
    it, rr, st = C.c_int(), C.c_double(), C.c_int()
    L.lpmx_solve_ex.argtypes = [C.c_int, C.c_double, C.c_double, C.c_int, C.c_double, C.c_int, C.POINTER(C.c_int),
                                C.POINTER(C.c_double), C.POINTER(C.c_int)]
    P.check(L.lpmx_solve_ex(prec, 1e-16, 0.0, 20000, 1e-2, 100, C.byref(it), C.byref(rr), C.byref(st)), "solve")
    assert st.value == 1
    return np.ascontiguousarray(get("DISP", (3 * n,)))


def residual(b, z):
    y = np.zeros_like(b)
    P.check(P.lib().lpmx_spmv(P.LPMX_FP64, P.ptr(z), P.ptr(y)), "product")
    return np.linalg.norm(b - y) / np.linalg.norm(b)


@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_bond_form_gives_way(prec, monkeypatch):
    L = P.lib()
    n, x, t, _ = P.build_sc_model(P.sc_box_for(28))
    b = tangent(n, t) * np.random.default_rng(1).standard_normal(3 * n)
    assert residual(b, solve(n, b, 0, prec)) <= 1.01e-8 and L.lpmx_bond_form_used() == 1
    monkeypatch.setenv("LPMX_MALLOC_TIGHT", "1")
    assert residual(b, solve(n, b, 1, prec)) <= 1.01e-8  # the hierarchy takes its room
    assert L.lpmx_bond_form_used() == 0
    tangent(n, t)
    assert residual(b, solve(n, b, 1, prec)) <= 1.01e-8 and L.lpmx_bond_form_used() == 0
    monkeypatch.delenv("LPMX_MALLOC_TIGHT")
    tangent(n, t)
    assert residual(b, solve(n, b, 1, prec)) <= 1.01e-8 and L.lpmx_bond_form_used() == 1
    P.check(L.lpmx_set_preconditioner(0), "default")


@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_cycle_without_its_dense_level(prec, monkeypatch):
    z, held = [], []
    for tight in (0, 1):
        monkeypatch.setenv("LPMX_MALLOC_TIGHT", str(tight))
        n, x, t, _ = P.build_sc_model(P.sc_box_for(16))
        b = tangent(n, t) * np.random.default_rng(1).standard_normal(3 * n)
        z.append(solve(n, b, 2, prec))
        lev, ts, by = C.c_int(), C.c_double(), C.c_int64()
        P.check(P.lib().lpmx_amg_info(C.byref(lev), C.byref(ts), C.byref(by)), "info")
        assert lev.value == 3
        held.append(by.value)
    P.check(P.lib().lpmx_set_preconditioner(0), "default")
    assert held[1] < held[0]
    # as one cycle against its restatement in test_gpu_dense_cycle.py
    assert np.abs(z[0] - z[1]).max() <= (1e-10 if prec == P.LPMX_FP64 else 1e-4) * np.abs(z[1]).max()
