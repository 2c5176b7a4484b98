"""Work items of the batched step: more items than wavefronts (tickets and the counter's reset), more
than 64 grids (the two-level search), one grid, and grids that finish at different attempts.  Each
grid must equal its own single-grid run bit for bit, state and control block."""
import numpy as np
import pytest
import torch

from clawpack_amd import _lib, problems
from clawpack_amd.batch import BatchedGrids
from clawpack_amd.device import make_desc

pytestmark = pytest.mark.gpu


def make(sizes, dtype, seg_h):
    d = make_desc(0, dtype, 64, 64, 0.1, 0.1, 3, 3, order=2, transverse_waves=2, mthlim=(4, 4, 4), bc_lower=(1, 2),
                  bc_upper=(1, 2), grav=1.0)
    grids = [problems.gaussian_humps(mx, my, 3 + k) for k, (mx, my) in enumerate(sizes)]
    b = BatchedGrids(d, grids, seg_h=seg_h)
    b.init(0.0, 1e-3, tend=0.02)
    return b


@pytest.mark.parametrize("name,sizes,seg_h,dtype", [
    ("one grid", [(70, 40)], 0, _lib.FP64),
    ("tickets", [(300, 200), (64, 64), (37, 190)], 1, _lib.FP64),
    ("tickets, many rounds", [(1200, 500), (61, 400)] * 3, 1, _lib.FP32),
    ("65 grids", [(20 + k, 30 + (7 * k) % 41) for k in range(65)], 0, _lib.FP64),
    ("130 grids", [(8 + k, 9 + (5 * k) % 23) for k in range(130)], 2, _lib.FP64),
])
def test_items_equal_single_grid_runs(name, sizes, seg_h, dtype):
    print("case batch items", name, flush=True)
    b, s = make(sizes, dtype, seg_h), make(sizes, dtype, 0)
    b.advance(5)
    b.advance(30)  # past tend for most grids
    s.advance_sequential(35)
    torch.cuda.synchronize()
    assert int(b.counter.item()) == 0
    cb, cs = b.read_ctrls(), s.read_ctrls()
    for g in range(len(sizes)):
        for f in ("t", "dt", "cfl", "cflmax", "numsteps", "attempts", "rejected", "cur", "done", "status", "arrive"):
            assert getattr(cb[g], f) == getattr(cs[g], f), (g, f)
        assert np.array_equal(b.download(g, cb), s.download(g, cs)), g
