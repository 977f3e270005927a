"""The crystal-plasticity return map on half a wavefront per particle, where its
branches can go wrong: particle counts that leave the last work-group part empty,
active sets on both sides of the eight whose Jacobian rows stay in registers, and a
hardening law and rate that take the general cosh, tanh and pow."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, oracle_model, push

pytestmark = pytest.mark.gpu

BASE = dict(tau0=10.0, taus=1e20, h0=100.0, q=1.0, eta=1.0, p=1.0, dtime=1.0, maxloop=20)


@pytest.fixture(scope="module")
def oracle():
    import oracle_py

    return oracle_py


def run_both(oracle, cp, box, amp):
    n = P.make_lattice(3, 0.5, box)
    L = P.lib()
    L.searchNormalNeighbor()
    L.searchAFEMNeighbor()
    x = P.field("XYZ", 3 * n).reshape(n, 3)
    t, c = P.sc_types(x), P.elastic_constants(70e3, 0.3)
    P.set_types(t, 5)
    P.set_materials([c] * 5, 1e30)
    P.set_params(plmode=1)
    P.set_cp_params(**cp)
    L.calcKnTv(), L.computedL(), L.slipSysDefine3D(), L.computeCab()
    m = oracle_model(oracle, x, 3, t, [c] * 5, plmode=1, sigmay=1e30, cp=cp)
    oracle.lib().orc_compute_cab(m.p)
    a = np.random.default_rng(5).standard_normal((3, 3))
    xd = x + x @ (amp * (a + a.T) / 2).T + 1e-4 * np.random.default_rng(6).standard_normal(x.shape)
    push("XYZ", xd)
    P.check(L.lpmx_bond_force(1), "plmode 1")
    fails = C.c_int()
    P.check(L.lpmx_cp_failures(C.byref(fails)), "failures")
    m.x[:] = xd
    oracle.lib().orc_bond_force_general(m.p, 1)
    assert fails.value == 0 and m.s.cp_fail == 0
    return n, m


FIELDS = (("CP_DA_SINGLE", "cp_dA_single"), ("CP_DGY", "cp_dgy"), ("CP_RSS", "cp_RSS"), ("CP_DA", "cp_dA"), ("F", "F"),
          ("PIN", "Pin"), ("STRESS", "stress"))


@pytest.mark.parametrize("h0,q,amp,most", [(100.0, 1.0, 2e-3, 8), (1e5, 0.0, 2e-3, 12), (3e5, 0.2, 1e-2, 9)])
def test_active_sets_around_the_register_rows(oracle, h0, q, amp, most):
    n, m = run_both(oracle, dict(BASE, h0=h0, q=q), [0, 6.5, 0, 4.3, 0, 5.1], amp)
    assert n % 4 == 1
    jact = get("CP_JACT", (n, 24))
    assert jact.sum(axis=1).max() == most
    np.testing.assert_array_equal(jact, m.cp_Jact)
    for name, ref in FIELDS:
        r = getattr(m, ref)
        np.testing.assert_array_equal(get(name, r.shape), r, err_msg=name)


def test_general_hardening_and_rate(oracle):
    # cosh, tanh and pow may differ from the host's by a unit in the last place; the slip
    # Jacobian's condition is below C_ab / h0 ~ 3e2, the loop at most 20 x 20 of them
    n, m = run_both(oracle, dict(BASE, h0=500.0, taus=60.0, p=0.9, eta=2.0), [0, 6.5, 0, 4.3, 0, 5.1], 2e-3)
    np.testing.assert_array_equal(get("CP_JACT", (n, 24)), m.cp_Jact)
    for name, ref in FIELDS:
        r = getattr(m, ref)
        assert np.abs(get(name, r.shape) - r).max() <= 400 * 3e2 * 2.3e-16 * max(1.0, np.abs(r).max()), name
