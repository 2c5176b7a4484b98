"""The reverse step where every interface of a wavefront is plain (subsonic, no entropy fix: the
shorter reverse form), where none is, and where a patch of fast flow mixes the two, against float64
autograd of the torch restatement.  Sizes: one and several segments of 58, the launch with 4 columns
per y workgroup and (from 512 workgroups) with 8, with a remainder of columns and rows in each.
Relative tolerance 1e-12, as for every reverse step.
"""
import numpy as np
import pytest
import torch

from clawpack_amd import _lib
from clawpack_amd.adjoint import adjoint_step
from clawpack_amd.device import make_desc
from oracle import torch_step as ts

pytestmark = pytest.mark.gpu


def state(mx, my, jet):
    rng = np.random.default_rng(mx + my)
    x, y = np.meshgrid((np.arange(mx) + 0.5) / mx, (np.arange(my) + 0.5) / my)
    w = lambda a: a * np.sin(2 * np.pi * (2 * x + y + rng.uniform())) * np.cos(2 * np.pi * (x - 3 * y + rng.uniform()))
    h, u, v = 1.0 + w(0.2), 0.05 + w(0.3), -0.02 + w(0.3)
    if jet:
        m = (np.abs(x - 0.4) < 0.1) & (np.abs(y - 0.6) < 0.15)
        u, v = u + np.where(m, 2.0 * np.cos(9 * y), 0.0), v + np.where(m, 1.7 * np.sin(11 * x), 0.0)
    return np.stack([h, h * u, h * v])


@pytest.mark.parametrize("shape", [(5, 4), (58, 61), (131, 73), (1030, 120)])
@pytest.mark.parametrize("lim", [1, 4])
@pytest.mark.parametrize("bc,jet", [((2, 2), False), ((3, 1), True)])
def test_reverse_step_plain_and_mixed(shape, lim, bc, jet):
    mx, my = shape
    print("case adjoint plain", shape, lim, bc, jet, flush=True)
    q = state(mx, my, jet)
    lam = np.random.default_rng(9).standard_normal(q.shape)
    dx, dy = 1.0 / mx, 1.2 / my
    dt = 0.15 * min(dx, dy)
    d = make_desc(0, _lib.FP64, mx, my, dx, dy, 3, 3, mthlim=(lim,) * 3, bc_lower=bc, bc_upper=bc, grav=1.0)
    got = adjoint_step(d, torch.tensor(q, device="cuda"), torch.tensor(lam, device="cuda"), dt).cpu().numpy()
    qt = torch.tensor(np.ascontiguousarray(q.transpose(0, 2, 1)), requires_grad=True)
    qn, _ = ts.step(qt, dt, dx, dy, "swe", 1.0, mthlim=(lim,) * 3, bc_lower=bc, bc_upper=bc, order=2,
                    transverse_waves=2)
    (qn * torch.tensor(np.ascontiguousarray(lam.transpose(0, 2, 1)))).sum().backward()
    ref = qt.grad.numpy().transpose(0, 2, 1)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
