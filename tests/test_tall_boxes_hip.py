"""Stencil boxes taller than a slab's 16-byte pieces reach.

On a tall grid whose feet spread over the column a tile's box spans well over a
hundred levels, more than one load of the wavefront's pieces covers; it must be
staged some other way and contracted at the places that way puts the levels.
Each case has such tiles (counted on the CPU from the oracle's feet) and must
give the direct-load kernels' doubles, for every parity of the rows.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.test_hip_parity import _random_case, cuda, make_plan
from tests.test_tile_boxes_hip import _predictors

pytestmark = pytest.mark.gpu

TILE = (4, 4, 16)
BOX_DOUBLES = 31104 // 8  # the smallest budget of the double tiles
PIECES = 64               # 16-byte pieces of one wavefront load


def tall_case(shape, lift, seed):
    """Feet a few cells apart in x and y and up to `lift` of the height in z."""
    c = _random_case(*shape, 4, "symmetric", seed=seed, cfl=1.0)
    nx, ny, nz = shape
    I, J = np.arange(nx + 2)[:, None, None], np.arange(ny + 2)[None, :, None]
    z = np.asarray(c["z_f"])[None, None, :] / c["Lz"]
    w = lift * c["Lz"] / c["dt"] * np.sin(np.pi * z) * np.cos(2.1 * I + 0.7) * np.cos(1.3 * J)
    u, v, _ = c["mids"]
    c["mids"] = [u, v, np.ascontiguousarray(w)]
    orc.apply_bc_all(*c["mids"])
    return c


def tall_tiles(c, depth=1.0):
    """Tiles whose box goes in slabs of rows of more than PIECES pieces."""
    P, h, tall = c["order"], c["order"] // 2 - 1, 0
    nx, ny, nz, dx, dy = c["nx"], c["ny"], c["nz"], c["Lx"] / c["nx"], c["Ly"] / c["ny"]
    sl = orc.SLOracle(nx, ny, nz, dx, dy, c["Lx"], c["Ly"], c["Lz"], c["z_f"], c["z_c"],
                      c["gamma"], stretching_type=c["stretching"], order=P)
    for comp, field, sx, sy in zip("uvw", c["fields"], (0.0, -0.5, -0.5), (-0.5, 0.0, -0.5)):
        shape = sl.arrival_shape(comp)
        xd, yd, zd = sl.departure(comp, *c["mids"], depth * c["dt"])
        k0 = sl.gather(comp, field, xd, yd, zd, want_index=True)[2][2]
        base = [np.floor(xd / dx + sx) - h, np.floor(yd / dy + sy) - h, k0]

        def extent(b):
            pad = [(0, -n % t) for n, t in zip(shape, TILE)]
            b = np.pad(b.reshape(shape).astype(np.int64), pad, mode="edge")
            b = b.reshape([q for n, t in zip(b.shape, TILE) for q in (n // t, t)])
            return b.max(axis=(1, 3, 5)) - b.min(axis=(1, 3, 5)) + P

        ex, ey, ez = map(extent, base)
        row = ez + (ez & 1)
        tall += int(((row > 2 * PIECES) & (ey * (row + 2) <= BOX_DOUBLES)
                     & (ex * ey * (row + 2) <= 8 * BOX_DOUBLES)).sum())
    return tall


@pytest.mark.parametrize("shape", [(24, 24, 256), (24, 22, 255), (23, 21, 240), (22, 25, 219)])
def test_tall_boxes_match_direct_loads(check, shape):
    c = tall_case(shape, 0.7, seed=sum(shape))
    for depth in (1.0, 2.0):
        n = tall_tiles(c, depth)
        check(f"tall boxes in slabs at depth {depth:g} dt", n > 0, f"{n} tiles")
    plan = make_plan(c, nu=1e-3)
    f = [cuda(a) for a in c["fields"]]
    m = [cuda(a) for a in c["mids"]]
    # U* = 2 V^n - V^{n-1} of the BDF2 predictor is the trajectory velocity
    before = [2.0 * a - b for a, b in zip(f, m)]
    res = {}
    for tile in (-1, 0):
        plan.set_option(plan.OPT_GATHER_TILE, tile)
        res[tile] = _predictors(plan, f, m, c["dt"])
        o = [torch.zeros(plan.shapes[k], dtype=torch.float64, device="cuda") for k in "uvw"]
        ncl = torch.zeros(1, dtype=torch.int64, device="cuda")
        plan.bdf2_predict(*f, *before, c["dt"], *o, ncl)
        res[tile]["bdf2 along the tall velocity"] = (o, int(ncl.item()))
        at = []
        for comp, fld in zip("uvw", f):
            x, y, z, v = (torch.empty(plan.n_arrival(comp), dtype=torch.float64, device="cuda")
                          for _ in range(4))
            plan.departure(comp, *m, c["dt"], x, y, z)
            plan.gather(comp, fld, x, y, z, v)
            at.append(v)
        res[tile]["gather at the feet"] = (at, 0)
    for name in res[0]:
        d = [(a - b).abs() for a, b in zip(res[0][name][0], res[-1][name][0])]
        check(f"{name}: tiled == direct", all(not bool(t.any()) for t in d)
              and res[0][name][1] == res[-1][name][1],
              f"{sum(int((t > 0).sum()) for t in d)} differ, max {max(float(t.max()) for t in d):.1e}")
