"""A block-Jacobi CG on an indefinite matrix stops with status 3 on the iterate before the
breakdown, on either side of the 1,024 slices up to which p.q is summed by the update's own
work-groups (343 and 1,077 slices here, and 8): against the same recurrence in numpy on the
exported matrix, shifted until its lowest modes are negative."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from lpm_harness import P, get, push

pytestmark = pytest.mark.gpu


def reference(A, n, b):
    i, j = A.row // 3, A.col // 3
    blocks = np.zeros((n, 3, 3))
    np.add.at(blocks, (i[i == j], A.row[i == j] % 3, A.col[i == j] % 3), A.data[i == j])
    minv, A = np.linalg.inv(blocks), A.tocsr()
    x, r = np.zeros(3 * n), b.copy()
    z = p = np.einsum("iab,ib->ia", minv, r.reshape(n, 3)).ravel()
    rz = r @ z
    for it in range(100):
        q = A @ p
        pq = p @ q
        if pq <= 0:
            assert pq < -1e-2 * np.linalg.norm(p) * np.linalg.norm(q)  # no matter of rounding
            return x, it
        x, r = x + rz / pq * p, r - rz / pq * q
        z = np.einsum("iab,ib->ia", minv, r.reshape(n, 3)).ravel()
        rz, old = r @ z, rz
        p = z + rz / old * p
    raise AssertionError("no breakdown")


@pytest.mark.parametrize("edge", [8, 28, 41])
@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_breakdown_keeps_the_last_iterate(edge, prec):
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
    IK = np.zeros(3 * n + 1, np.int32)
    JK, K = np.zeros(n * 64 * 9, np.int32), np.zeros(n * 64 * 9)
    P.check(L.lpmx_export_upper_csr(P.ptr(IK), P.ptr(JK), P.ptr(K)), "export")
    rows = np.repeat(np.arange(3 * n), np.diff(IK))
    nk = len(rows)
    JK, K = JK[:nk] - 1, np.ascontiguousarray(K[:nk])
    diag = (JK == rows) & (dbc.ravel()[rows] == 1)
    K[diag] -= 0.1 * K[diag].mean()
    P.check(L.lpmx_import_upper_csr(P.ptr(K)), "import")
    U = sp.csr_matrix((K, (rows, JK)), shape=(3 * n, 3 * n))
    ref, iters = reference((U + sp.triu(U, 1).T).tocoo(), n, b)
    assert iters >= 3
    P.check(L.lpmx_set_preconditioner(0), "block-Jacobi")
    it, rr, st = C.c_int(), C.c_double(), C.c_int()
    L.lpmx_solve_ex.argtypes = [C.c_int, C.c_double, C.c_double, C.c_int, C.c_double, C.c_int, C.POINTER(C.c_int),
                                C.POINTER(C.c_double), C.POINTER(C.c_int)]
    P.check(L.lpmx_solve_ex(prec, 1e-16, 0.0, 1000, 1e-2, 100, C.byref(it), C.byref(rr), C.byref(st)), "solve")
    assert st.value == 3 and it.value == iters
    z = get("DISP", (3 * n,))
    err = np.abs(z - ref).max() / np.abs(ref).max()
    print(f"{edge} {prec}: {iters} iterations, off by {err:.2e}", flush=True)
    # rounding (1.1e-16, 6e-8) of sums of 59 blocks, amplified at each of the few steps by
    # |p| |K p| / p.q, here below 1e2 at the last ones
    assert err <= (1e-11 if prec == P.LPMX_FP64 else 1e-3)
