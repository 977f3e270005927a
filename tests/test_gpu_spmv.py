"""The sliced SpMV (16 or 4 wavefronts per slice) on tangents of every lattice: row counts
below and around the 64 of a slice, rows of 17 to 61 blocks, both value precisions."""
import numpy as np
import pytest

from lpm_harness import P, push

pytestmark = pytest.mark.gpu


def box(lattice, m):
    return [0.0, m + 0.2, 0.0, 4.3, 0.0, 1.0] if lattice < 2 else [0.0, m + 0.2, 0.0, 3.2, 0.0, 2.3]


@pytest.mark.parametrize("lattice", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("m", [2, 5, 9, 17])
def test_sliced_spmv(lattice, m):
    L = P.lib()
    n = P.make_lattice(lattice, 0.5, box(lattice, m))
    L.searchNormalNeighbor()
    nk = L.searchAFEMNeighbor()
    d = 2 if lattice < 2 else 3
    x = P.field("XYZ", 3 * n).reshape(n, 3)
    P.set_types(np.zeros(n, np.int32), 1)
    P.set_materials([P.elastic_constants(200e3, 0.3)], 200.0)
    P.set_params(plmode=0)
    L.calcKnTv()
    rng = np.random.default_rng(m)
    push("XYZ", x + 1e-3 * rng.standard_normal(x.shape) * (np.arange(3) < d))
    P.check(L.lpmx_tangent(), "tangent")
    IK, JK, K = np.zeros(d * n + 1, np.int32), np.zeros(nk, np.int32), np.zeros(nk)
    P.check(L.lpmx_export_upper_csr(P.ptr(IK), P.ptr(JK), P.ptr(K)), "export")
    rows, cols = np.repeat(np.arange(d * n), np.diff(IK)), JK - 1
    A = np.zeros((d * n, d * n))
    A[rows, cols] = K
    A[cols, rows] = K
    v, y = rng.standard_normal(d * n), np.zeros(d * n)
    # sums of at most 61 * d products: 200 units in the last place of the absolute row sum
    bound = np.abs(A) @ np.abs(v)
    P.check(L.lpmx_spmv(P.LPMX_FP64, P.ptr(v), P.ptr(y)), "spmv")
    assert (np.abs(y - A @ v) <= 200 * 1.2e-16 * bound).all()
    # FP32 values, FP64 vectors and sums: half a unit in the last place of each value
    P.check(L.lpmx_spmv(P.LPMX_MIXED, P.ptr(v), P.ptr(y)), "spmv32")
    assert (np.abs(y - A @ v) <= 6.1e-8 * bound).all()
