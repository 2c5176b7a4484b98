"""Step kernels with the limiter and the transverse mode fixed at compile time, against the oracle:
every solver, limiter and mode, split and not, at sizes of one strip and several with odd edges; and a
batch, which runs the general kernel for superbee and van Leer, against single-grid runs.

FP64: max|dq| <= 1e-12 max|q|; FP32 to the rounding of its inputs and sums (5e-6 of max|q|)."""
import numpy as np
import pytest

from clawpack_amd import _lib, problems
from clawpack_amd.batch import BatchedGrids
from clawpack_amd.device import DeviceGrid, make_desc
from oracle import corc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [_lib.FP64, _lib.FP32])
@pytest.mark.parametrize("lim", [1, 2, 3, 4])
@pytest.mark.parametrize("tw", [0, 1, 2])
@pytest.mark.parametrize("solver", ["swe", "euler"])
def test_unsplit(solver, tw, lim, dtype):
    for mx, my in ((60, 5), (131, 67)):
        print("case limiter kernels", solver, tw, lim, dtype, mx, my, flush=True)
        q = problems.random_smooth_swe(mx, my, 4) if solver == "swe" else problems.random_euler(mx, my, 2)
        if dtype == _lib.FP32:
            q = q.astype(np.float32).astype(np.float64)
        neq, dx, dy, dt = q.shape[0], 0.1, 0.13, 0.02
        d = corc.make_desc(solver, mx, my, dx, dy, grav=1.0, gamma=1.4, order=2, transverse_waves=tw,
                           mthlim=(lim,) * 4)
        qo, cflo = corc.step_hyperbolic(d, corc.make_ctrl(bc_lower=(3, 1), bc_upper=(3, 1)), q, dt)
        g = DeviceGrid(make_desc(0 if solver == "swe" else 1, dtype, mx, my, dx, dy, neq, neq, order=2,
                                 transverse_waves=tw, mthlim=(lim,) * neq, bc_lower=(3, 1), bc_upper=(3, 1),
                                 grav=1.0, gamma=1.4))
        g.init_ctrl(0.0, dt)
        g.upload(q)
        cfl, c = g.step(dt)
        assert c.status == 0
        tol = 1e-12 if dtype == _lib.FP64 else 5e-6
        assert np.abs(g.download() - qo).max() <= tol * np.abs(q).max()
        assert abs(cfl - cflo) <= (1e-13 if dtype == _lib.FP64 else 5e-6) * cflo


@pytest.mark.parametrize("lim,tw", [(2, 2), (3, 1), (4, 0)])
def test_batch_equals_single_grids(lim, tw):
    print("case limiter kernels, batch", lim, tw, flush=True)
    sizes = [(70, 40), (121, 33), (64, 200)]
    runs = []
    for _ in range(2):
        d = make_desc(0, _lib.FP64, 64, 64, 0.1, 0.1, 3, 3, order=2, transverse_waves=tw, mthlim=(lim,) * 3,
                      bc_lower=(1, 2), bc_upper=(1, 2), grav=1.0)
        b = BatchedGrids(d, [problems.gaussian_humps(mx, my, 3 + k) for k, (mx, my) in enumerate(sizes)])
        b.init(0.0, 1e-3, target_steps=20)
        runs.append(b)
    runs[0].advance(12)
    runs[1].advance_sequential(12)
    for g in range(len(sizes)):
        assert np.array_equal(runs[0].download(g), runs[1].download(g)), g
