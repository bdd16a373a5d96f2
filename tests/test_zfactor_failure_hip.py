"""A z-solve that is refused leaves no table behind that passes for built.

nz = 6142: a column of u is one element too long for LDS, a column of w just
fits.  The joined call refuses u; solving w on its own afterwards, with the same
(dt, theta), must give what a fresh plan gives.
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["implicit_project", "zsolve"])
def test_refused_solve_leaves_no_table(check, first):
    c = _random_case(3, 2, 6142, 4, "symmetric", seed=5, cfl=0.5)
    f = [cuda(t) for t in c["fields"]]
    out = []
    for refused in (False, True):
        plan = make_plan(c, nu=1e-2)
        if refused:
            g = [t.clone() for t in f]
            with pytest.raises(RuntimeError):
                if first == "zsolve":
                    plan.zsolve("u", g[0], 0.01, 1.0)
                else:
                    plan.implicit_project(*g, 0.01, 1.0, 0.01, 0.01)
            check("nothing solved", all(map(torch.equal, f, g)), "fields changed")
            with pytest.raises(RuntimeError):
                plan.zsolve("u", g[0], 0.01, 1.0)
        w = f[2].clone()
        plan.zsolve("w", w, 0.01, 1.0)
        out.append(w)
    check("w after a refused call == w of a fresh plan", torch.equal(*out),
          f"max {float((out[0] - out[1]).abs().max()):.1e}")
    check("w solved", not torch.equal(out[0], f[2]), "unchanged")
