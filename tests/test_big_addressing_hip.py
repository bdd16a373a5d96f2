"""Tile and feet kernels with 64-bit addresses.

A plane of 2^24 elements or more takes the kernels built with 64-bit addresses
and 32-bit index products.  Three thin planes reach that in little memory: the
step passes, the split passes, departure and gather (with feet far apart too,
which the second pass gathers) must give the direct-load kernels' doubles, and
an ensemble's member those of its own run.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

NX, NY = 3, 59049  # rows of a plane odd in number


def _nz(order):
    """(NY + 2)(nz + 2) > 2^24; rows of u and v odd, or those of w."""
    return 283 if order == 4 else 284


def _config(order, storage):
    nz = _nz(order)
    return {"grid": {"nx": NX, "ny": NY, "nz": nz},
            "domain": {"Lx": float(NX), "Ly": float(NY), "Lz": float(nz)},
            "flow": {"Re": 1000.0, "U_bulk": 1.0, "gamma": 1.2},
            "sl": {"interp_order": order,
                   "interp_dtype": "fp32_accum64" if storage == 32 else "fp64"}}


def _fields(shapes, seed):
    """Smooth in z and y with noise of a tenth, about a cell a unit of time."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for q, c in enumerate("uvw"):
        s = shapes[c]
        i, j, k = (torch.arange(n, dtype=torch.float64, device="cuda") for n in s)
        f = torch.randn(s, dtype=torch.float64, device="cuda", generator=gen).mul_(0.1)
        f += torch.sin(0.21 * j + q)[:, None] * torch.cos(0.05 * k + q)[None, :]
        f += (0.3 * torch.cos(2 * math.pi * i / NX + q))[:, None, None]
        out.append(f.mul_((1.0, 0.8, 0.5)[q]))
    return out


def _same(check, tag, a, b):
    n = sum(int((x != y).sum()) for x, y in zip(a, b))
    check(tag, n == 0, f"{n} differ")


@pytest.mark.parametrize("order", [4, 6])
def test_thick_planes_match_direct_loads(check, order):
    from slchannel_amd import SLChannelFlow

    print(f"{NX}x{NY}x{_nz(order)} order {order}", flush=True)
    flow = SLChannelFlow(config=_config(order, 64))
    plan = flow.plan
    f, m = _fields(flow.shapes, 1), _fields(flow.shapes, 2)
    plan.apply_bc(*f)
    plan.apply_bc(*m)
    ncl = torch.zeros(1, dtype=torch.int64, device="cuda")

    def star():
        return [torch.zeros(flow.shapes[c], dtype=torch.float64, device="cuda") for c in "uvw"]

    def calls(fused=1):
        plan.set_option(plan.OPT_BDF2_FUSED, fused)
        yield "advect", lambda o: plan.advect(*f, *m, 1.3, *o, ncl)
        yield "bdf1", lambda o: plan.bdf1_predict(*f, 1.3, *o, ncl)
        yield "bdf2", lambda o: plan.bdf2_predict(*f, *m, 0.7, *o, ncl)
        yield "high CFL", lambda o: plan.advect(*f, *m, 9.0, *o, ncl)

    for fused in (1, 0):
        for name, call in calls(fused):
            print(f"  {name}, fused {fused}", flush=True)
            res = []
            for tile in (-1, 0):
                plan.set_option(plan.OPT_GATHER_TILE, tile)
                ncl.zero_()
                o = star()
                call(o)
                res.append((o, int(ncl.item())))
            _same(check, f"{name}, fused {fused}: tiled == direct", res[0][0], res[1][0])
            check(f"{name}: clamped feet", res[0][1] == res[1][1], f"{res[0][1]} {res[1][1]}")
            if fused == 0:
                continue
            if name in ("advect", "high CFL"):
                dt = 1.3 if name == "advect" else 9.0
                first = {"u": (slice(1, None), slice(1, -1)), "v": (slice(1, -1), slice(1, None)),
                         "w": (slice(1, -1), slice(1, -1))}
                for c, fld, s in zip("uvw", f, res[0][0]):
                    n = plan.n_arrival(c)
                    x, y, z = (torch.empty(n, dtype=torch.float64, device="cuda")
                               for _ in range(3))
                    plan.departure(c, *m, dt, x, y, z)
                    got = torch.empty(n, dtype=torch.float64, device="cuda")
                    plan.gather(c, fld, x, y, z, got, None)
                    nzi = plan.arrival_shape(c)[2]
                    want = s[first[c]][..., 1:1 + nzi]
                    _same(check, f"{name} {c}: departure + gather == direct advect",
                          [got.view(want.shape)], [want])
    del f, m, flow, plan
    torch.cuda.empty_cache()


@pytest.mark.parametrize("order,storage", [(4, 32), (6, 64)])
def test_thick_member_matches_its_own_run(check, order, storage):
    from slchannel_amd import SLChannelFlow
    from slchannel_amd.ensemble import Ensemble

    print(f"member {NX}x{NY}x{_nz(order)} order {order} storage {storage}", flush=True)
    cfg, dt = _config(order, storage), 0.8
    flow = SLChannelFlow(config=cfg)
    flow.set_fields(*_fields(flow.shapes, 3))
    flow.apply_bc_uvw()
    flow.project_initial()
    init = [t.clone() for t in (flow.u, flow.v, flow.w, flow.p)]
    for _ in range(3):
        flow.step_sl_bdf2(dt)
    alone = [t.cpu() for t in (flow.u, flow.v, flow.w, flow.p)]
    del flow
    torch.cuda.empty_cache()
    ens = Ensemble(order=order, storage=storage)
    mid = ens.add(cfg, dt, fields=init)
    small = dict(cfg, grid={"nx": 12, "ny": 10, "nz": 14},
                 domain={"Lx": 12.0, "Ly": 10.0, "Lz": 14.0})
    ens.add(small, dt)
    for _ in range(3):
        ens.step()
    got = ens.get_fields(mid)
    _same(check, "member == its own run", [got[k].cpu() for k in "uvwp"], alone)
    ens.close()
    torch.cuda.empty_cache()
