"""Neighbour lists by a wavefront per particle: partners, shells and first lengths against
the oracle, bit for bit, on particle counts that do and do not fill a work-group of 16
particles, lattices of one and of few cells, in 3D and 2D, and on shuffled positions."""
import numpy as np
import pytest

from lpm_harness import P, get, host_lattice, oracle_model, sc_pair

pytestmark = pytest.mark.gpu


def check(n, nb, m):
    np.testing.assert_array_equal(get("NB_INITIAL", (n,)), m.nb_initial)
    np.testing.assert_array_equal(get("NEIGHBORS", (n, nb)), m.nbr)
    live = m.nbr >= 0
    np.testing.assert_array_equal(get("NSIGN", (n, nb))[live], m.nsign[live])
    np.testing.assert_array_equal(get("DISTANCE_INITIAL", (n, nb))[live], m.L0[live])


@pytest.mark.parametrize("edge", [2, 3, 5, 6])  # 8, 27, 125 and 216 particles
def test_sc(oracle, edge):
    _, n, x, t, m = sc_pair(oracle, edge)
    check(n, 18, m)


@pytest.mark.parametrize("ly", [1.0, 4.0, 9.0])
def test_hex(oracle, ly):
    L = P.lib()
    n = P.make_lattice(1, 0.5, [0, 14.0, 0, ly, 0, 1.0])
    L.searchNormalNeighbor()
    x = P.positions()
    c = P.elastic_constants(70e3, 0.25)
    m = oracle_model(oracle, x, 1, np.zeros(n, np.int32), [c])
    check(n, 12, m)


def test_shuffled_positions(oracle):
    box = [0, 7.0, 0, 6.0, 0, 5.0]
    x = oracle.create_lattice(2, 0.5, box)
    x = np.ascontiguousarray(x[np.random.default_rng(4).permutation(len(x))])
    n, _ = host_lattice(oracle, 2, 0.5, box, x)
    L = P.lib()
    L.searchNormalNeighbor()
    c = P.elastic_constants(200e3, 0.3)
    m = oracle_model(oracle, x, 2, np.zeros(n, np.int32), [c])
    check(n, 18, m)
