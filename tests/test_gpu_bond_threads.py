"""The per-bond kernels of the J2 and elastic laws on lists of 8, 12, 14 and 18 slots
(square, hexagonal, BCC, FCC), particle counts that leave the last work-group part
empty, broken and damaged bonds, and a particle range: bit-exact with the oracle."""
import numpy as np
import pytest

from lpm_harness import P, get, oracle_model, push

pytestmark = pytest.mark.gpu

BOXES = {0: [0.0, 10.0, 0.0, 8.5, 0.0, 1.0], 1: [0.0, 12.0, 0.0, 10.0, 0.0, 1.0], 3: [0.0, 5.2, 0.0, 4.3, 0.0, 3.1],
         4: [0.0, 5.2, 0.0, 4.3, 0.0, 6.1]}


@pytest.fixture(scope="module")
def oracle():
    import oracle_py

    return oracle_py


@pytest.mark.parametrize("lattice", [0, 1, 3, 4])
@pytest.mark.parametrize("mode", [0, 6])
def test_bond_threads_bit_exact(oracle, lattice, mode):
    L = P.lib()
    n = P.make_lattice(lattice, 0.5, BOXES[lattice])
    L.searchNormalNeighbor()
    L.searchAFEMNeighbor()
    x = P.field("XYZ", 3 * n).reshape(n, 3)
    t, c = np.zeros(n, np.int32), P.elastic_constants(200e3, 0.3)
    P.set_types(t, 1)
    P.set_materials([c], 200.0)
    P.set_params(plmode=mode, J2_H=2000.0, J2_xi=0.3)
    L.calcKnTv()
    L.computedL()
    m = oracle_model(oracle, x, lattice, t, [c], plmode=mode, sigmay=200.0, J2_H=2000.0, J2_xi=0.3)
    nb = m.nbr.shape[1]
    assert n % 32 != 0 and nb == {0: 8, 1: 12, 3: 18, 4: 14}[lattice]
    rng = np.random.default_rng(lattice)
    dim = 2 if lattice < 2 else 3
    xd = x + 2e-3 * rng.standard_normal(x.shape) * (np.arange(3) < dim)
    has = m.nbr >= 0
    # broken on both sides with weight 0, as the damage rules leave bonds: the reference
    # evaluates a particle with its unbroken partners only
    i, j = np.minimum(np.arange(n)[:, None], m.nbr), np.maximum(np.arange(n)[:, None], m.nbr)
    broken = has & ((i * 7919 + j * 104729) % 11 == 0)
    fields = {"XYZ": (xd, "x"), "J2_BETA0": (3.0 * rng.standard_normal((n, 6)), None),
              "J2_ALPHA0": (1e-3 * rng.uniform(size=n), None),
              "DLP0": (2e-5 * rng.standard_normal((n, nb)) * has, None),
              "DAMAGE_BROKEN": (np.where(broken, 0.0, 1.0), "dmg_broken"),
              "DAMAGE_W": (np.where(broken, 0.0, rng.uniform(0.5, 1.0, (n, nb))), "dmg_w"),
              "NB": (m.nb - broken.sum(axis=1).astype(np.int32), "nb")}
    for name, (v, ref) in fields.items():
        push(name, np.ascontiguousarray(v))
        if ref:
            getattr(m, ref)[:] = v
    m.beta[:, :, 0], m.alpha[:, 0] = fields["J2_BETA0"][0], fields["J2_ALPHA0"][0]
    m.dLp[:, :, 0] = fields["DLP0"][0]
    P.check(L.lpmx_bond_force_range(mode, 0, n), "bond force")
    P.check(L.lpmx_compute_stress(), "stress")
    oracle.lib().orc_bond_force_general(m.p, mode)
    for name, ref in (("DL", m.dL), ("F", m.F), ("PIN", m.Pin), ("STRESS", m.stress)):
        np.testing.assert_array_equal(get(name, ref.shape), ref, err_msg=name)
    # a range writes its own particles' forces only
    push("PIN", np.full(3 * n, 7.0))
    P.check(L.lpmx_bond_force_range(mode, 5, 40), "range")
    pin = get("PIN", (n, 3))
    np.testing.assert_array_equal(pin[5:45], m.Pin.reshape(n, 3)[5:45])
    assert (pin[:5] == 7.0).all() and (pin[45:] == 7.0).all()
