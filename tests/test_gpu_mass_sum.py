"""The compensated mass sum against the correctly rounded sum (math.fsum of the stored values), at the
edges of its launch forms: one block or many, a remainder of the 16-byte vectors, planes that are
not 16-byte aligned (odd cell counts, component 1 and 2), and values that cancel.

Tolerance: a compensated sum of n terms is off by at most eps |S| + 2 n eps^2 sum|x|, with one
rounding more for the final addition.
"""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from clawpack_amd import _lib
from clawpack_amd.device import DeviceGrid, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("mx,my", [(2, 2), (3, 5), (128, 128), (127, 129), (128, 129), (181, 181), (1024, 512),
                                   (1025, 513), (2047, 1031)])
def test_mass_sum_edges(dtype, mx, my):
    print("case mass sum", dtype, mx, my, flush=True)
    rng = np.random.default_rng(mx * 7 + my)
    q = rng.standard_normal((3, my, mx)) * np.exp(rng.uniform(-20, 20, (3, my, mx)))
    g = DeviceGrid(make_desc(0, dtype, mx, my, 0.1, 0.1, 3, 3))
    g.set_planes(torch.from_numpy(q).to(g.torch_dtype))
    stored = g.planes().to(torch.float64).cpu().numpy()
    eps, n = 2.0 ** -53, mx * my
    for m in range(3):
        ref = math.fsum(stored[m].ravel().tolist())
        tol = 2 * eps * abs(ref) + 2 * n * eps ** 2 * float(np.abs(stored[m]).sum())
        v = g.mass_sum(m)
        assert abs(v - ref) <= tol, (m, v, ref)
        assert g.mass_sum(m) == v
        out = torch.zeros(1, dtype=torch.float64, device=g.device)
        assert g.lib.claw2d_mass_sum_noalloc(C.byref(g.desc), C.c_void_p(g.planes().data_ptr()), m,
                                             C.c_void_p(out.data_ptr()), None) == 0
        torch.cuda.synchronize()
        assert out.item() == v
