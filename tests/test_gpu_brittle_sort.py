"""The brittle selection sorts its candidates by the reference's gap sequence on all of them
at once: the bonds broken, their order and ties included, against the oracle, for the
smallest candidate lists, lists around a power of two and a work-group, and a long one."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, get, oracle_model, push

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bonds", [1, 2, 31, 32, 33, 127, 128, 129, 513, 900])
@pytest.mark.parametrize("nbreak", [1, 20])
def test_selection(oracle, bonds, nbreak):
    L = P.lib()
    n = P.make_lattice(1, 0.5, [0, 14.0, 0, 12.0, 0, 1.0])
    L.searchNormalNeighbor()
    L.searchAFEMNeighbor()
    x = P.positions()
    P.set_types(np.zeros(n, np.int32), 1)
    c = P.elastic_constants(70e3, 0.25)
    P.set_materials([c], 200.0)
    P.set_params(plmode=6, critical_bstrain=1e-3, nbreak=nbreak)
    L.calcKnTv()
    m = oracle_model(oracle, x, 1, np.zeros(n, np.int32), [c], plmode=6, critical_bstrain=1e-3, nbreak=nbreak)
    rng = np.random.default_rng(bonds)
    pairs = [(i, a) for i in range(n) for a in range(m.nb_initial[i]) if m.nbr[i, a] > i]
    s = np.zeros((n, 12))
    for q in rng.permutation(len(pairs))[:bonds]:
        i, a = pairs[q]
        j = m.nbr[i, a]
        # few distinct values: many ties
        s[i, a] = s[j, list(m.nbr[j]).index(i)] = 1.1e-3 + 1e-4 * rng.integers(0, 9)
    dl = np.where(m.nbr >= 0, s * m.L0, 0.0)
    push("DL", dl)
    P.check(L.lpmx_set_params(C.byref(P.Params(6, 0.0, 0.0, 0.5, 0.9, 0.0, 1e-3, nbreak))), "params")
    k = C.c_int()
    P.check(L.lpmx_damage(6, C.byref(k)), "brittle")
    m.dL[:] = dl
    bi, bj = np.zeros(2 * bonds, np.int32), np.zeros(2 * bonds, np.int32)
    ko = oracle.lib().orc_damage_brittle(m.p, oracle.ptr(bi), oracle.ptr(bj), 2 * bonds)
    assert k.value == ko == 2 * bonds
    np.testing.assert_array_equal(get("DAMAGE_BROKEN", (n, 12)), m.dmg_broken)
    gi, gj, cnt = np.zeros(2 * bonds, np.int32), np.zeros(2 * bonds, np.int32), C.c_int()
    P.check(L.lpmx_get_broken(P.ptr(gi), P.ptr(gj), 2 * bonds, C.byref(cnt)), "broken")
    q = cnt.value
    assert q == min(nbreak, ko)
    np.testing.assert_array_equal(gi[:q], bi[:q])
    np.testing.assert_array_equal(gj[:q], bj[:q])
