"""step_imex updates flow.u, v, w where they are.

A caller that keeps the field tensors across IMEX steps (a monitor, a writer, a
statistics loop) reads the current fields in them, and a run of this scheme
alone holds no second set of fields.  The steps must give the doubles of their
separate calls, ghosts and the stored right-hand sides included, with columns in
the lanes' registers and (nz 1030) in LDS.
"""

import math

import numpy as np
import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu


def _flow(shape, top):
    from slchannel_amd import SLChannelFlow

    nx, ny, nz = shape
    f = SLChannelFlow(config={
        "grid": {"nx": nx, "ny": ny, "nz": nz},
        "domain": {"Lx": 4 * math.pi, "Ly": 2 * math.pi, "Lz": 2.0},
        "flow": {"Re": 2000.0, "U_bulk": 1.0, "gamma": 1.5},
        "boundary_conditions": {"top_wall": {"type": top}}, "sl": {"interp_order": 4}})
    rng = np.random.default_rng(sum(shape))
    f.set_fields(*(1.0 * (c == "u") + 0.1 * rng.standard_normal(f.shapes[c]) for c in "uvw"))
    f.project_initial()
    return f


@pytest.mark.parametrize("shape,top", [((7, 5, 9), "dirichlet"), ((24, 20, 66), "neumann"),
                                       ((12, 9, 257), "dirichlet"), ((6, 4, 1030), "neumann")])
def test_held_fields_follow_the_steps(check, shape, top):
    f, dt = _flow(shape, top), 1e-4
    held = [f.u, f.v, f.w]
    # the separate calls, on fields of their own
    plan = _flow(shape, top).plan
    g, prev = [t.clone() for t in held], None
    p = torch.zeros_like(f.p)
    for n in range(3):
        ub, fo = f.step_imex(dt)
        plan.apply_bc(*g)
        r = [torch.zeros_like(t) for t in g]
        plan.imex_rhs(*g, *r)
        plan.ab2_update(*g, r, prev, dt)
        prev = r
        plan.apply_bc(*g)
        for comp, t in zip("uvw", g):
            plan.zsolve(comp, t, dt, 0.5)
        plan.apply_bc(*g)
        plan.project_step(*g, dt, dt, p)
        out = torch.empty(4, dtype=torch.float64, device="cuda")
        plan.bulk_force(*g, f.U_bulk, dt, out)
        same = all(a is b for a, b in zip((f.u, f.v, f.w), held))
        check(f"step {n + 1}: the fields' own tensors", same, "rebound")
        check(f"step {n + 1}: held fields are the new ones", all(map(torch.equal, held, g)),
              f"max {max(float((a - b).abs().max()) for a, b in zip(held, g)):.1e}")
        check(f"step {n + 1}: pressure, bulk", torch.equal(f.p, p) and ub.item() == out[2].item()
              and fo.item() == out[1].item(), "")
        check(f"step {n + 1}: stored rhs, zero off the interior",
              all(map(torch.equal, f._imex_prev, r)), "")
    check("no second set of fields", f._star is None, "")


@pytest.mark.parametrize("theta,nu", [(0.5, 0.0), (0.5, 1e-2), (0.75, 1e-2)])
@pytest.mark.parametrize("nz", [6, 65, 520, 1030])
def test_plan_step_matches_separate_calls(check, theta, nu, nz):
    """Any theta below 1, inviscid too (no explicit part, still another source)."""
    c = _random_case(7, 6, nz, 4, "symmetric", seed=nz, cfl=0.5)
    plan, dt = make_plan(c, nu=nu), 0.01
    a = [cuda(t) for t in c["fields"]]
    b = [t.clone() for t in a]
    r, s = ([torch.zeros_like(t) for t in a] for _ in range(2))
    prev = [torch.randn_like(t) for t in a]
    plan.imex_rhs(*a, *r)
    plan.ab2_update(*a, r, prev, dt)
    plan.implicit_project(*a, dt, theta, dt, dt)
    plan.imex_step(*b, s, prev, dt, theta)
    check("fields", all(map(torch.equal, a, b)),
          f"max {max(float((x - y).abs().max()) for x, y in zip(a, b)):.1e}")
    check("rhs", all(map(torch.equal, r, s)), "")
    for bad in (0.0, 1.0):
        with pytest.raises(RuntimeError):
            plan.imex_step(*b, s, prev, dt, bad)
