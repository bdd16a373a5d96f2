"""The joined implicit and projection part of a step against its separate calls.

slc_implicit_project solves the three components' z-columns in one launch, reads
no ghost entry (x and y wrapped, w's wall faces zero) and writes every ghost with
the interior value it follows; the bulk shift does the same for u.  Ghost fills,
slc_zsolve and slc_project_step in turn must give the very same doubles, ghosts
included, at every split of a column over the lanes.
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu


# unknowns per lane of (u and v, w): equal and one class apart (nz one past a
# multiple of 64), the shortest columns, and columns past the lanes' registers
@pytest.mark.parametrize("theta", [1.0, 0.5])
@pytest.mark.parametrize("shape,top", [
    ((8, 6, 3), "dirichlet"), ((3, 5, 17), "neumann"), ((34, 33, 31), "dirichlet"),
    ((12, 10, 64), "neumann"), ((12, 10, 65), "dirichlet"), ((6, 7, 129), "dirichlet"),
    ((6, 5, 257), "neumann"), ((5, 4, 513), "dirichlet"), ((4, 3, 1030), "dirichlet")])
def test_joined_calls_match_separate_calls(check, theta, shape, top):
    c = _random_case(*shape, 4, "symmetric", seed=sum(shape), cfl=0.5)
    plan = make_plan(c, nu=1e-2, top=top)
    dt = 0.01
    a = [cuda(t) for t in c["fields"]]
    b = [t.clone() for t in a]
    pa = torch.zeros(plan.shapes["p"], dtype=torch.float64, device="cuda")
    pb = torch.full_like(pa, float("nan"))
    plan.apply_bc(*a)
    for comp, t in zip("uvw", a):
        plan.zsolve(comp, t, dt, theta)
    plan.apply_bc(*a)
    plan.project_step(*a, dt, dt, pa)
    plan.implicit_project(*b, dt, theta, dt, dt, pb)
    for name, x, y in zip("uvwp", a + [pa], b + [pb]):
        check(f"{name} after the projection", torch.equal(x, y), "doubles differ")
    # nothing left for a ghost fill to change
    filled = [t.clone() for t in b]
    plan.apply_bc(*filled)
    check("ghosts after the projection", all(map(torch.equal, b, filled)), "fill changes them")
    ra = torch.empty(4, dtype=torch.float64, device="cuda")
    for rep in range(3):
        plan.bulk_force(*b, 1.0 + rep, dt, ra)
        filled = b[0].clone()
        plan.apply_bc(filled, b[1], b[2])
        check(f"u's ghosts after shift {rep}", torch.equal(b[0], filled), "fill changes them")
        mean = torch.empty(4, dtype=torch.float64, device="cuda")
        plan.bulk_velocity(b[0], mean)
        check(f"mean after shift {rep}", mean[3].item() == ra[2].item(),
              f"{mean[3].item()} {ra[2].item()}")
