"""The joined IMEX pass refuses outputs that share an array with its inputs.

Its points read their neighbours' old values while other points are written, so
any field given as an output too would be a race.  The previous rhs may be the
new one's array: each point reads its own entry before it writes it.
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan

pytestmark = pytest.mark.gpu


def test_shared_arrays_are_refused(check):
    c = _random_case(6, 6, 8, 4, "symmetric", seed=3, cfl=0.5)
    plan = make_plan(c, nu=1e-2)

    def array(like=None):  # room for any component in each
        buf = torch.zeros(1024, dtype=torch.float64, device="cuda")
        return buf if like is None else buf[:like.numel()].view(like.shape).copy_(like)

    f = [array(cuda(t)) for t in c["fields"]]
    plan.apply_bc(*f)
    ptr, stream = plan._lib.slc_imex_advance, plan._stream()

    def call(new, r, prev):
        return ptr(plan._h, *(t.data_ptr() for t in f + new + r + prev), 0.01, stream)

    def fresh():
        return [array() for _ in "uvw"]

    before = [t.clone() for t in f]
    for i in range(6):
        for j in range(3):
            out = fresh() + fresh()
            out[i] = f[j]
            check(f"output {i} = field {j} refused", call(out[:3], out[3:], fresh()) != 0, "")
        for j in range(i):
            out = fresh() + fresh()
            out[i] = out[j]
            check(f"output {i} = output {j} refused", call(out[:3], out[3:], fresh()) != 0, "")
    torch.cuda.synchronize()
    check("nothing written", all(map(torch.equal, f, before)), "fields changed")
    prev = [torch.randn_like(t) for t in f]
    a, ra = ([torch.zeros_like(t) for t in f] for _ in range(2))
    b, rb = [torch.zeros_like(t) for t in f], [t.clone() for t in prev]
    plan.imex_advance(*f, a, ra, prev, 0.01)
    plan.imex_advance(*f, b, rb, rb, 0.01)
    inner = {"u": (slice(1, None), slice(1, -1), slice(1, -1)),
             "v": (slice(1, -1), slice(1, None), slice(1, -1)),
             "w": (slice(1, -1), slice(1, -1), slice(1, -1))}
    check("previous rhs in place of the new one", all(
        torch.equal(x[inner[k]], y[inner[k]]) for p, q in ((a, b), (ra, rb))
        for k, x, y in zip("uvw", p, q)), "doubles differ")
