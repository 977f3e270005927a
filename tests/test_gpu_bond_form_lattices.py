"""The products over the bonds on lists of 14 slots (BCC, the run-time slot count) and 18
(FCC) above 20,000 particles, against the stored tangent, which a repeated elimination
returns to: one V-cycle, and the iterate after three CG steps.  With a bond whose shell puts
a two-hop partner outside the pattern, the stored tangent throughout."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, push

pytestmark = pytest.mark.gpu

BOX = {3: [0.0, 25.2, 0.0, 25.0, 0.0, 25.4], 4: [0.0, 26.2, 0.0, 26.0, 0.0, 26.4]}


def build(lattice):
    L = P.lib()
    n = P.make_lattice(lattice, 0.5, BOX[lattice])
    L.searchNormalNeighbor()
    L.searchAFEMNeighbor()
    x = P.field("XYZ", 3 * n).reshape(n, 3)
    P.set_types(np.zeros(n, np.int32), 1)
    P.set_materials([P.elastic_constants(200e3, 0.3)], 200.0)
    P.set_params(plmode=0, J2_H=2000.0, J2_xi=0.0)
    L.calcKnTv()
    L.computedL()
    nb = P.gint("nneighbors").value
    assert n > 20000 and n % 64 != 0 and nb == {3: 18, 4: 14}[lattice]
    rng = np.random.default_rng(lattice)
    nbr = get("NEIGHBORS", (n, nb))
    push("DLP0", np.ascontiguousarray(np.where(nbr >= 0, rng.uniform(-1e-4, 1e-4, (n, nb)), 0.0)))
    push("XYZ", np.ascontiguousarray(x + rng.uniform(-1e-4, 1e-4, (n, 3))))
    dbc = np.ones((n, 3), np.int32)
    dbc[x[:, 2] < x[:, 2].min() + 1.0] = 0
    dbc[x[:, 2] > x[:, 2].max() - 1.0, 2] = 0
    return n, nb, nbr, dbc


def solves(n, b, prec):
    """One V-cycle's correction and three CG steps' iterate on the current matrix."""
    L = P.lib()
    L.lpmx_solve_ex.argtypes = [C.c_int, C.c_double, C.c_double, C.c_int, C.c_double, C.c_int, C.POINTER(C.c_int),
                                C.POINTER(C.c_double), C.POINTER(C.c_int)]
    out = []
    for kind, maxit, want in ((2, 10, 1), (0, 3, 2)):
        push("RESIDUAL", b)
        P.check(L.lpmx_set_preconditioner(kind), "preconditioner")
        it, rr, st = C.c_int(), C.c_double(), C.c_int()
        P.check(L.lpmx_solve_ex(prec, 1e-16, 0.0, maxit, 1e-16, 1, C.byref(it), C.byref(rr), C.byref(st)), "solve")
        assert st.value == want
        out.append(get("DISP", (3 * n,)).copy())
    return out


@pytest.mark.parametrize("lattice", [3, 4])
@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_products(lattice, prec):
    L = P.lib()
    n, _, _, dbc = build(lattice)
    P.check(L.lpmx_tangent(), "tangent")
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    b = np.random.default_rng(1).standard_normal(3 * n) * dbc.ravel()
    L.lpmx_bc_eliminate_ex.argtypes = [C.c_int]
    P.check(L.lpmx_bc_eliminate_ex(1), "eliminate")
    assert L.lpmx_bond_form_used() == 1
    got = solves(n, b, prec)
    P.check(L.lpmx_bc_eliminate_ex(1), "eliminate again: the same matrix, of a later version")
    assert L.lpmx_bond_form_used() == 0
    ref = solves(n, b, prec)
    P.check(L.lpmx_set_preconditioner(0), "default")
    for name, z, r in zip(("cycle", "CG"), got, ref):
        err = np.abs(z - r).max() / np.abs(r).max()
        print(f"lattice {lattice} {prec} {name}: {err:.2e}", flush=True)
        # as in test_gpu_bond_form.py: rounding of sums of up to 61 blocks or 36 bond terms,
        # through a cycle or through three steps
        assert err <= (1e-12 if prec == P.LPMX_FP64 else 2e-5)


def test_partner_outside_the_pattern():
    L = P.lib()
    n, nb, nbr, dbc = build(3)
    i = n // 2
    ns = get("NSIGN", (n, nb))
    e = int(np.flatnonzero(ns[i] == 0)[0])
    j = nbr[i, e]
    ns[i, e] = ns[j, list(nbr[j]).index(i)] = 1
    push("NSIGN", ns)
    P.check(L.lpmx_tangent(), "tangent")
    push("DISPBC_INDEX", np.ascontiguousarray(dbc.ravel()))
    P.check(L.lpmx_bc_eliminate(), "eliminate")
    assert L.lpmx_bond_form_used() == 0
