"""The LDS tiles' ways of staging a stencil box against the direct-load kernels.

A tile's box goes to LDS whole or in slabs of planes, in 16-byte pieces whose
place in a row turns with the parity of the row (odd row lengths, odd or even
periods), in 4-byte pieces where a wrapped box breaks those turns, or not at
all when no plane fits.  Every way adds the same products in the same order, so
the doubles must be the direct kernels' (SLC_OPT_GATHER_TILE = -1) for every
parity of the grid's lengths, at small and at large displacements.
"""

import numpy as np
import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu


def _predictors(plan, f, m, dt):
    out = {}
    for name in ("advect", "bdf1", "bdf2"):
        o = [torch.zeros(plan.shapes[k], dtype=torch.float64, device="cuda") for k in "uvw"]
        ncl = torch.zeros(1, dtype=torch.int64, device="cuda")
        if name == "advect":
            plan.advect(*f, *m, dt, *o, ncl)
        elif name == "bdf1":
            plan.bdf1_predict(*f, dt, *o, ncl)
        else:
            plan.bdf2_predict(*f, *m, dt, *o, ncl)
        out[name] = (o, int(ncl.item()))
    return out


# every parity of (nx, ny, nz); rows shorter than a box (nz 5, 7); boxes past
# the LDS budget (slabs, then none) as the displacement grows
@pytest.mark.parametrize("order", [4, 6])
@pytest.mark.parametrize("shape,cfl", [
    ((20, 18, 22), 1.0), ((20, 18, 33), 1.0), ((20, 19, 22), 1.0), ((20, 19, 33), 1.0),
    ((21, 18, 33), 1.0), ((21, 19, 33), 1.0), ((21, 19, 22), 4.0), ((20, 18, 40), 4.0),
    ((21, 19, 41), 6.0), ((17, 16, 70), 9.0), ((33, 30, 7), 2.0), ((9, 8, 5), 1.0),
    ((40, 38, 34), 60.0)])
def test_staged_boxes_match_direct_loads(check, order, shape, cfl):
    c = _random_case(*shape, order, "symmetric", seed=sum(shape) + order, cfl=cfl)
    plan = make_plan(c, nu=1e-3)
    f = [cuda(a) for a in c["fields"]]
    m = [cuda(a) for a in c["mids"]]
    plan.set_option(plan.OPT_GATHER_TILE, -1)
    ref = _predictors(plan, f, m, c["dt"])
    plan.set_option(plan.OPT_GATHER_TILE, 0)
    got = _predictors(plan, f, m, c["dt"])
    # the same fields 8 bytes past a 16-byte boundary: the pieces of every row
    # start one level earlier or later
    shifted = []
    for a in f:
        buf = torch.empty(a.numel() + 1, dtype=torch.float64, device="cuda")
        shifted.append(buf[1:].view(a.shape))
        shifted[-1].copy_(a)
    off = _predictors(plan, shifted, m, c["dt"])
    for name in ref:
        for tag, res in (("", got), (" at an 8-byte offset", off)):
            same = all(torch.equal(x, y) for x, y in zip(res[name][0], ref[name][0]))
            dev = max((x - y).abs().max().item() for x, y in zip(res[name][0], ref[name][0]))
            check(f"{name}{tag}: tiled == direct", same and res[name][1] == ref[name][1],
                  f"max|d|={dev:.1e} ncl={res[name][1]},{ref[name][1]}")


@pytest.mark.parametrize("order", [4, 6])
def test_far_and_non_finite_feet_match_direct_loads(check, order):
    """Feet many periods outside the domain, and NaN and infinite ones among
    ordinary feet: the same values (NaN where the direct gather gives NaN)."""
    c = _random_case(24, 20, 22, order, "symmetric", seed=3, cfl=1.0)
    plan = make_plan(c)
    rng = np.random.default_rng(9)
    for ic, comp in enumerate("uvw"):
        n = plan.n_arrival(comp)
        xd, yd = (rng.uniform(0, L, n) for L in (c["Lx"], c["Ly"]))
        zd = rng.uniform(0, c["Lz"], n)
        far = rng.random(n) < 0.01
        xd[far] += rng.choice([-1e6, 40.0, 1e9], far.sum()) * c["Lx"]
        bad = rng.random(n) < 0.01
        xd[bad] = rng.choice([np.nan, np.inf, -np.inf], bad.sum())
        zd[rng.random(n) < 0.01] = np.nan
        args = [cuda(a) for a in (c["fields"][ic], xd, yd, zd)]
        outs = []
        for tile in (-1, 0):
            plan.set_option(plan.OPT_GATHER_TILE, tile)
            o = torch.zeros(n, dtype=torch.float64, device="cuda")
            plan.gather(comp, *args, o)
            outs.append(o)
        check(f"{comp}: tiled == direct", torch.equal(outs[0].isnan(), outs[1].isnan()) and
              torch.equal(outs[0].nan_to_num(), outs[1].nan_to_num()),
              f"{int(outs[0].isnan().sum())} NaN values")
