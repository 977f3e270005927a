"""The reverse sweep by a thread per bond on lists of 18 (FCC) and 14 (BCC, run-time slot
count) slots, particle counts that leave the last work-group part empty, against the
oracle's."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, oracle_model, push

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oracle():
    import oracle_py

    return oracle_py


@pytest.mark.parametrize("lattice,box", [(3, [0.0, 5.2, 0.0, 4.3, 0.0, 3.1]), (4, [0.0, 5.2, 0.0, 4.3, 0.0, 6.1])])
def test_vjp_matches_oracle(oracle, lattice, box):
    L = P.lib()
    n = P.make_lattice(lattice, 0.5, box)
    L.searchNormalNeighbor()
    L.searchAFEMNeighbor()
    x = P.field("XYZ", 3 * n).reshape(n, 3)
    assert n % 32
    t, c = np.zeros(n, np.int32), P.elastic_constants(200e3, 0.3)
    P.set_types(t, 1)
    P.set_materials([c], 200.0)
    P.set_params(plmode=0, J2_H=2000.0, J2_xi=0.3)
    L.calcKnTv()
    L.computedL()
    m = oracle_model(oracle, x, lattice, t, [c], plmode=0, sigmay=200.0, J2_H=2000.0, J2_xi=0.3)
    rng = np.random.default_rng(lattice)
    nb, live = m.nbmax, m.nbr >= 0
    xd = x + 5e-4 * rng.standard_normal((n, 3))
    dlp = 1e-5 * rng.standard_normal((n, nb)) * live
    beta, alpha = 5.0 * rng.standard_normal((n, 6)), 1e-3 * rng.uniform(0, 1, n)
    P.check(L.lpmx_set_params(C.byref(P.Params(0, 2000.0, 0.3, 0.5, 0.9, 0.0, 1e-2, 20))), "params")
    for name, v in (("XYZ", xd), ("DLP0", dlp), ("J2_BETA0", beta), ("J2_ALPHA0", alpha)):
        push(name, v)
    m.x[:], m.dLp[:, :, 0], m.beta[:, :, 0], m.alpha[:, 0] = xd, dlp, beta, alpha
    seeds = [rng.standard_normal(3 * n), np.ascontiguousarray(rng.standard_normal((n, nb)) * live * 1e5),
             np.ascontiguousarray(rng.standard_normal((n, 6))), rng.standard_normal(n) * 1e3]
    outs = lambda: [np.zeros(3 * n), np.zeros((n, nb)), np.zeros((n, 6)), np.zeros(n), np.zeros(n), np.zeros(n)]  # noqa: E731
    dev, ref, hb, hr = outs(), outs(), np.zeros(1), C.c_double()
    P.check(L.lpmx_vjp(*[P.ptr(s) for s in seeds], *[P.ptr(o) for o in dev], P.ptr(hb)), "vjp")
    oracle.lib().orc_eval_j2(m.p)
    assert m.pl_flag.sum() > 0
    oracle.lib().orc_vjp_j2(m.p, *[oracle.ptr(s) for s in seeds], *[oracle.ptr(o) for o in ref], C.byref(hr))
    for name, a, b in zip(["positions", "dLp0", "beta0", "alpha0", "modulus", "sigmay"], dev, ref):
        assert np.abs(b).max() > 0, name
        # sums of at most 36 products of rounded factors, some cancelling: 1e-11 as the SC test
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max(), name
    assert abs(hb[0] - hr.value) <= 1e-11 * abs(hr.value)
