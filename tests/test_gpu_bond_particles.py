"""The one-thread-per-particle kernels of the J2 and elastic laws (from 100,000 particles on)
on the broken and weighted bonds, the particle range and the lists of 8 to 18 slots of
test_gpu_bond_threads.py: bit-exact with the oracle."""
import functools

import pytest

import test_gpu_bond_threads as small

pytestmark = pytest.mark.gpu

BOXES = {0: [0.0, 321.0, 0.0, 323.0, 0.0, 1.0], 1: [0.0, 300.0, 0.0, 302.0, 0.0, 1.0],
         3: [0.0, 40.2, 0.0, 41.3, 0.0, 44.1], 4: [0.0, 42.2, 0.0, 43.3, 0.0, 43.1]}


@pytest.mark.parametrize("lattice", [0, 1, 3, 4])
@pytest.mark.parametrize("mode", [0, 6])
def test_bond_particles_bit_exact(oracle, lattice, mode, monkeypatch):
    monkeypatch.setattr(small, "BOXES", BOXES)
    monkeypatch.setattr(oracle.Model, "setup", functools.partialmethod(oracle.Model.setup, cells=True))
    small.test_bond_threads_bit_exact(oracle, lattice, mode)
    assert small.P.gint("nparticle").value >= 100000
