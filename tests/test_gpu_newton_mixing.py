"""The V-cycle Newton loop with the mixing solved on the device: depths from none to the
largest reach one solution, and differences down at the rounding floor (a Gram matrix
that is singular to working precision) leave the iterate where it is."""
import numpy as np
import pytest

from lpm_harness import P, get, tol_for

pytestmark = pytest.mark.gpu


def run(prec, depth, tol=1e-11, maxit=3000, edge=7):
    n, x, _, _ = P.build_sc_model(P.sc_box_for(edge), sigmay=200.0, H=20000.0)
    steps = P.sc_uniaxial_steps(edge - 1.0, np.array([0.9e-3, 1.5e-3]))
    s = P.solver(precision=prec, rtol2=1e-8, atol2=0.0, maxit=1000, newton_tol=tol, newton_maxit=maxit,
                 accel_depth=depth, precond=2)
    rc, out = P.run_steps(steps, s)
    return rc, out, get("XYZ", (n, 3)) - x


@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
@pytest.mark.parametrize("depth", [0, 1, 2, 31])
def test_depths_reach_one_solution(prec, depth):
    rc, out, u = run(prec, depth)
    rr, _, ur = run(P.LPMX_FP64, 32)
    assert rc == 0 and rr == 0, [(o.status, o.newton_iters) for o in out]
    assert np.abs(u - ur).max() <= tol_for(prec) * np.abs(ur).max() * 10  # Newton 1e-11, times the condition of K
    assert (sum(o.accel_mixed for o in out) > 0) == (depth > 0)


@pytest.mark.parametrize("prec", [P.LPMX_FP64, P.LPMX_MIXED])
def test_mixing_at_the_rounding_floor(prec):
    _, _, ur = run(P.LPMX_FP64, 32)
    rc, out, u = run(prec, 32, tol=0.0, maxit=150)  # iterates on, far below the last residual
    assert rc == -6 and np.isfinite(u).all()
    # positions of order 10 rounded to 1.8e-15, over a displacement of 1e-2, times 1e3 of
    # the stretch-to-position amplification and the accelerated steps between
    assert np.abs(u - ur).max() <= 1e-8 * np.abs(ur).max()
