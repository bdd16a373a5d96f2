"""slc_imex_advance, rhs and AB2 update in one pass, against the two calls.

Both walk the grid along x with two planes in registers; grids of one run and of
several, runs that end short, odd rows and the smallest grids must all give the
doubles of slc_imex_rhs and slc_ab2_update on the interiors and leave every
other entry alone.
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu

INNER = {"u": (slice(1, None), slice(1, -1), slice(1, -1)),
         "v": (slice(1, -1), slice(1, None), slice(1, -1)),
         "w": (slice(1, -1), slice(1, -1), slice(1, -1))}


@pytest.mark.parametrize("shape", [(1, 2, 4), (3, 5, 7), (16, 12, 20), (33, 17, 64),
                                   (70, 96, 130), (131, 65, 254)])
def test_advance_matches_rhs_and_update(check, shape):
    c = _random_case(*shape, 4, "symmetric", seed=sum(shape), cfl=0.5)
    plan = make_plan(c, nu=1e-2)
    f = [cuda(t) for t in c["fields"]]
    plan.apply_bc(*f)
    prev = [torch.randn_like(t) for t in f]
    dt = 0.01
    for rp in (None, prev):
        r = [torch.full_like(t, float("nan")) for t in f]
        plan.imex_rhs(*f, *r)
        new = [t.clone() for t in f]
        plan.ab2_update(*new, r, rp, dt)
        mark = [torch.full_like(t, 7.0) for t in f]
        rm = [torch.full_like(t, 7.0) for t in f]
        plan.imex_advance(*f, mark, rm, rp, dt)
        for k, a, b, ra, rb in zip("uvw", new, mark, r, rm):
            s = INNER[k]
            check(f"{k} new", torch.equal(a[s], b[s]), "doubles differ")
            check(f"{k} rhs", torch.equal(ra[s], rb[s]), "doubles differ")
            check(f"{k} rhs finite", bool(torch.isfinite(ra).all()), "entries left unwritten")
            for t in (b, rb):
                t[s] = 7.0
                check(f"{k} others", bool((t == 7.0).all()), "written outside the interior")
