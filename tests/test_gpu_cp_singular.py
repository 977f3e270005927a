"""A slip Jacobian with an exact zero pivot ends its particle's return map on all of the
particle's lanes: the failure count and everything that the evaluation leaves of a failed
particle and of its neighbours are the oracle's, bit for bit.  The zero is at the first pivot (no stiffness
at all) or at the second (all systems alike), for every particle or for some of them, so
that the two particles of a wavefront part ways."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, oracle_model, push
from test_gpu_cp_lanes import BASE, FIELDS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pivot", [1, 2])
@pytest.mark.parametrize("share", [1.0, 0.4])
def test_singular_slip_jacobian(oracle, pivot, share):
    # no hardening and no rate: the Jacobian is the active part of C_ab
    cp = dict(BASE, h0=0.0, eta=0.0)
    n = P.make_lattice(3, 0.5, [0, 6.5, 0, 4.3, 0, 5.1])
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
    cab = m.cp_Cab.reshape(n, 24 * 24)
    rng = np.random.default_rng(2)
    hit = rng.uniform(size=n) < share
    cab[hit] = 0.0 if pivot == 1 else cab.max()
    # the other particles keep theirs, made well conditioned on every active set
    cab[~hit] += 0.5 * cab.max() * np.eye(24).ravel()
    push("CP_CAB", cab)
    a = np.random.default_rng(5).standard_normal((3, 3))
    xd = x + x @ (2e-3 * (a + a.T) / 2).T + 1e-4 * np.random.default_rng(6).standard_normal(x.shape)
    push("XYZ", xd)
    P.check(L.lpmx_bond_force(1), "plmode 1")
    fails = C.c_int()
    P.check(L.lpmx_cp_failures(C.byref(fails)), "failures")
    m.x[:] = xd
    oracle.lib().orc_bond_force_general(m.p, 1)
    jact = get("CP_JACT", (n, 24))
    assert fails.value == m.s.cp_fail and 0 < fails.value <= hit.sum()
    assert (jact[hit].sum(axis=1) == pivot).any() and (share == 1.0 or (jact[~hit].sum(axis=1) > 2).any())
    np.testing.assert_array_equal(jact, m.cp_Jact)
    for name, ref in FIELDS + (("DL", "dL"), ("DDLP", "ddLp")):
        r = getattr(m, ref)
        np.testing.assert_array_equal(get(name, r.shape), r, err_msg=name)
    for name, ref in (("DLP2", m.dLp), ("CP_GY2", m.cp_gy), ("CP_A2", m.cp_A)):
        np.testing.assert_array_equal(get(name, ref.shape[:-1]), ref[..., 2], err_msg=name)
