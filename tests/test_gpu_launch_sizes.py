"""The default cut of a launch at the ends of its rule: one-row segments, half and all SIMDs, two and
more wavefronts per SIMD, grids of one strip and of one segment.  Segments are launch shape only, so
the default must equal explicit segment heights bit for bit (state and CFL number)."""
import numpy as np
import pytest
import torch

from clawpack_amd import _lib, problems
from clawpack_amd.device import DeviceGrid, make_desc

pytestmark = pytest.mark.gpu


def step(q, dx, dy, dtype, split, lim, seg_h):
    mx, my = q.shape[1], q.shape[2]
    d = make_desc(0, dtype, mx, my, dx, dy, 3, 3, order=2, transverse_waves=2, mthlim=(lim,) * 3,
                  bc_lower=(3, 1), bc_upper=(3, 1), grav=1.0, seg_h=seg_h)
    g = DeviceGrid(d, "cuda:0", split=split)
    g.upload(q)
    g.init_ctrl(0.0, 1e-4)
    cfl, c = g.step(0.2 * min(dx, dy))
    assert c.status == 0 and np.isfinite(cfl)
    return g.q[g.cur].cpu(), cfl


@pytest.mark.parametrize("mx,my", [(2, 2), (61, 3), (59, 700), (2000, 5), (300, 300), (640, 480), (1023, 777)])
@pytest.mark.parametrize("dtype,split,lim", [(_lib.FP64, False, 4), (_lib.FP64, True, 1), (_lib.FP32, False, 3)])
def test_default_cut_equals_explicit_segments(mx, my, dtype, split, lim):
    print("case launch sizes", mx, my, dtype, split, lim, flush=True)
    q, dx, dy = problems.gaussian_humps(mx, my, 5)
    ref, cref = step(q, dx, dy, dtype, split, lim, 0)
    for seg in (1, 2, 23):
        got, cgot = step(q, dx, dy, dtype, split, lim, seg)
        assert cgot == cref, seg
        assert torch.equal(got, ref), seg
