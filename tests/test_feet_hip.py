"""Feet of the departure call against the direct-load advect kernel.

The feet are traced with the step kernels' sampling (32-bit addresses, one round
of loads a sample); slc_advect with the tiles off traces them with located
intervals and gathers at once.  Gathering at the stored feet must give the same
doubles and the same clamp count, from ghost-shaped fields and from packed node
buffers, for every grid parity, number of iterations and displacement (points
that leave the domain by more than a period included).
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda

pytestmark = pytest.mark.gpu


def _plan(c, iters):
    from slchannel_amd import HipPlan

    return HipPlan(int(c["nx"]), int(c["ny"]), int(c["nz"]), float(c["Lx"]), float(c["Ly"]),
                   float(c["Lz"]), c["z_f"], c["z_c"], float(c["gamma"]),
                   stretching_type=str(c["stretching"]), order=int(c["order"]),
                   n_traj_iters=iters)


@pytest.mark.parametrize("stretching", ["symmetric", "bottom"])
@pytest.mark.parametrize("shape,cfl,iters", [
    ((20, 18, 22), 1.0, 2), ((21, 19, 33), 2.5, 1), ((9, 8, 5), 1.0, 3), ((17, 16, 70), 9.0, 2),
    ((33, 30, 7), 2.0, 0), ((40, 38, 65), 200.0, 2)])
def test_feet_match_direct_advect(check, stretching, shape, cfl, iters):
    c = _random_case(*shape, 4, stretching, seed=sum(shape), cfl=cfl)
    c.setdefault("stretching", stretching)
    plan = _plan(c, iters)
    plan.set_option(plan.OPT_GATHER_TILE, -1)
    f = [cuda(a) for a in c["fields"]]
    m = [cuda(a) for a in c["mids"]]
    plan.apply_bc(*f)
    plan.apply_bc(*m)
    star = [torch.zeros_like(t) for t in f]
    ncl = torch.zeros(1, dtype=torch.int64, device="cuda")
    plan.advect(*f, *m, c["dt"], *star, ncl)
    # node buffers: the unique nodes, ghost levels included
    first = {"u": (slice(1, None), slice(1, -1)), "v": (slice(1, -1), slice(1, None)),
             "w": (slice(1, -1), slice(1, -1))}
    base = {"u": (0, 1), "v": (1, 0), "w": (1, 1)}
    nodes = [t[base[k][0]:base[k][0] + plan.nx, base[k][1]:base[k][1] + plan.ny].contiguous()
             for k, t in zip("uvw", m)]
    for layout, traj in ((0, m), (1, nodes)):
        count = torch.zeros(1, dtype=torch.int64, device="cuda")
        for k, fld, s in zip("uvw", f, star):
            n = plan.n_arrival(k)
            x, y, z = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(3))
            plan.departure(k, *traj, c["dt"], x, y, z, nclamp=count, layout=layout)
            out = torch.empty(n, dtype=torch.float64, device="cuda")
            plan.gather(k, fld, x, y, z, out, None)
            nzi = plan.arrival_shape(k)[2]
            want = s[first[k]][..., 1:1 + nzi]
            check(f"{k} layout {layout}", torch.equal(out.reshape(want.shape), want),
                  f"{(out.reshape(want.shape) != want).sum().item()} differ")
        check(f"clamp count layout {layout}", int(count.item()) == int(ncl.item()),
              f"{int(count.item())} {int(ncl.item())}")
