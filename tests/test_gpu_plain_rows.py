"""Rows whose interfaces are all plain (subsonic both ways, no entropy fix) take a shorter form of
the interface arithmetic, chosen per wavefront and row; the others take the general form.  The two
are the same bit for bit, so a result cannot depend on which columns share a wavefront: a state
with a patch of transonic and supersonic flow in a subsonic sea, rolled along x and y, gives the
rolled result, for shifts that move the patch across strips (60 columns), segments and the grid's
edges.  Against the oracle the step is held to 1e-12 max|q| (FP64), as every step is.
"""
import numpy as np
import pytest

from clawpack_amd import problems
from clawpack_amd.device import DeviceGrid, make_desc
from oracle import corc

pytestmark = pytest.mark.gpu
MX, MY = 150, 70


def patch_state(solver):
    """(q, aux): smooth subsonic flow with a jet patch, faster than the waves, and its edges."""
    rng = np.random.default_rng(5)
    x, y = np.meshgrid((np.arange(MX) + 0.5) / MX, (np.arange(MY) + 0.5) / MY, indexing="ij")
    w = lambda a: a * np.sin(2 * np.pi * (2 * x + y + rng.uniform())) * np.cos(2 * np.pi * (x - 3 * y + rng.uniform()))
    jet = (np.abs(x - 0.37) < 0.06) & (np.abs(y - 0.55) < 0.12)
    h, u, v = 1.0 + w(0.2), 0.2 + w(0.2), -0.1 + w(0.2)
    u = u + np.where(jet, 2.5 * np.cos(9 * y), 0.0)
    v = v + np.where(jet, 2.0 * np.sin(11 * x), 0.0)
    if solver == "euler":
        p = 1.0 + w(0.2)
        return np.stack([h, h * u, h * v, p / 0.4 + 0.5 * h * (u * u + v * v)]), None
    b = -1.2 + w(0.3) if solver == "bathy" else None
    return np.stack([h, h * u, h * v]), None if b is None else b[None]


def step(solver, dtype, split, tw, lim, q, aux, dt, seg_h):
    sid = {"swe": 0, "euler": 1, "bathy": 2}[solver]
    neq = q.shape[0]
    d = make_desc(sid, dtype, MX, MY, 1.0 / MX, 1.0 / MY, neq, neq, transverse_waves=tw, mthlim=(lim,) * 4,
                  bc_lower=(2, 2), bc_upper=(2, 2), grav=1.0, gamma=1.4, seg_h=seg_h)
    g = DeviceGrid(d, split=split)
    g.upload(q)
    if aux is not None:
        g.upload_aux(aux)
    g.init_ctrl(0.0, dt)
    cfl, _ = g.step(dt)
    return g.download(), cfl


@pytest.mark.parametrize("solver", ["swe", "euler", "bathy"])
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("split,tw,lim", [(False, 2, 4), (False, 1, 1), (False, 0, 3), (True, 2, 4)])
def test_plain_and_general_rows_agree_bitwise(solver, dtype, split, tw, lim):
    print("case plain rows", solver, dtype, split, tw, lim, flush=True)
    q, aux = patch_state(solver)
    dt = 0.2 / MX
    ref, cfl = step(solver, dtype, split, tw, lim, q, aux, dt, 0)
    od = corc.make_desc(solver, MX, MY, 1.0 / MX, 1.0 / MY, grav=1.0, gamma=1.4, transverse_waves=tw,
                        mthlim=(lim,) * 4, **({"num_aux": 1, "fwave": 1, "dry_tolerance": 1e-3}
                                              if solver == "bathy" else {}))
    kw = {"dimensional_split": split}
    if solver == "bathy":
        kw.update(aux_bc_lower=(2, 2), aux_bc_upper=(2, 2))
    oc = corc.make_ctrl(bc_lower=(2, 2), bc_upper=(2, 2), **kw)
    if dtype == 0:
        qo, cflo = corc.step_hyperbolic(od, oc, q, dt, **({"aux": aux} if aux is not None else {}))
        assert np.abs(ref - qo).max() <= 1e-12 * np.abs(q).max()
        assert abs(cfl - cflo) <= 1e-13 * cflo
    for sx, sy, seg in ((17, 0, 0), (61, 23, 5), (-30, 41, 16), (95, -9, 70)):
        rq = np.roll(q, (sx, sy), axis=(1, 2))
        ra = None if aux is None else np.roll(aux, (sx, sy), axis=(1, 2))
        out, c = step(solver, dtype, split, tw, lim, rq, ra, dt, seg)
        assert c == cfl
        assert np.array_equal(np.roll(out, (-sx, -sy), axis=(1, 2)), ref), (sx, sy, seg)
