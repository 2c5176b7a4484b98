"""Limiters of the general kernel against the oracle where their forms can go wrong: waves of zero
strength, subnormal and very small strengths beside ordinary ones, single and mixed ids.

Bar as for every step: max|dq| <= 1e-12 max|q| in FP64; FP32 against the same step in FP64 to the
rounding of its inputs and sums (2e-6 of max|q|)."""
import numpy as np
import pytest

from clawpack_amd import problems
from clawpack_amd.device import DeviceGrid, make_desc
from oracle import corc

pytestmark = pytest.mark.gpu


def state(mx, my, scale):
    q = problems.random_smooth_swe(mx, my, 3)
    q[:, : mx // 3, :] = np.array([1.0, 0.0, 0.0])[:, None, None]  # at rest: every strength is 0
    rng = np.random.default_rng(7)
    q[1:, mx // 8: mx // 4, :] = scale * rng.standard_normal((2, mx // 4 - mx // 8, my))
    return q


@pytest.mark.parametrize("scale", [0.0, 5e-324, 1e-310, 1e-300, 1e-160, 1e-20])
@pytest.mark.parametrize("lim", [(3, 3, 3), (2, 2, 2), (3, 4, 3), (1, 3, 5)])
@pytest.mark.parametrize("dtype", [0, 1])
def test_small_strengths(scale, lim, dtype):
    mx, my, dx, dy, dt = 67, 35, 0.1, 0.1, 0.015
    print("case limiter forms", scale, lim, dtype, flush=True)
    q = state(mx, my, scale)
    if dtype == 1:
        q = q.astype(np.float32).astype(np.float64)
    d = corc.make_desc("swe", mx, my, dx, dy, grav=1.0, gamma=1.4, order=2, transverse_waves=2, mthlim=lim + (0,))
    qo, cflo = corc.step_hyperbolic(d, corc.make_ctrl(bc_lower=(1, 1), bc_upper=(1, 1)), q, dt)
    g = DeviceGrid(make_desc(0, dtype, mx, my, dx, dy, 3, 3, order=2, transverse_waves=2, mthlim=lim,
                             bc_lower=(1, 1), bc_upper=(1, 1), grav=1.0))
    g.init_ctrl(0.0, dt)
    g.upload(q)
    cfl, c = g.step(dt)
    got = g.download()
    assert c.status == 0 and np.isfinite(got).all()
    tol = 1e-12 if dtype == 0 else 2e-6
    assert np.abs(got - qo).max() <= tol * np.abs(q).max()
    assert abs(cfl - cflo) <= (1e-13 if dtype == 0 else 2e-6) * cflo
