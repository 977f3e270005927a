"""lpmx_update_rr_noalloc at the largest model that it serves and one particle above."""
import ctypes as C

import numpy as np
import pytest

from lpm_harness import P, push
from test_zz_no_alloc import both

pytestmark = pytest.mark.gpu

LARGEST = 1048576


def model(n):
    L = P.lib()
    x = np.zeros((n, 3))
    x[:, 0] = np.arange(n)
    d = P.ModelDesc(3, 2, n, 18, 6, 12, 60, 0.5, 1.0, 2**0.5, 1.0)
    P.check(L.lpmx_model_create(C.byref(d), P.ptr(x)), "model")
    rng = np.random.default_rng(1)
    push("PIN", rng.standard_normal(3 * n))
    push("PEX", rng.standard_normal(3 * n))
    dbc = (rng.uniform(size=3 * n) > 0.2).astype(np.int32)
    push("DISPBC_INDEX", dbc)
    return dbc


def test_largest_model():
    dbc = model(LARGEST)
    (a, b, c, r1), (a2, b2, c2, r2) = both(LARGEST)
    assert (a2, b2, c2) == (a, b, c) and c == (dbc == 0).sum() and a > 0 and b > 0
    np.testing.assert_array_equal(r2, r1)
    model(LARGEST + 1)
    a = C.c_double()
    assert P.lib().lpmx_update_rr_noalloc(C.byref(a), None, None) == -2
    P.check(P.lib().lpmx_model_destroy(), "destroy")
