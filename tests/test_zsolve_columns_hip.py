"""Wavefronts that solve many z-columns against wavefronts that solve one.

A grid of more columns than the chip holds wavefronts has each of them walk
several, with the factorisation, the scans' products and the level distances'
reciprocals formed once.  The columns of a small grid, one to a wavefront, must
come out as the same doubles, at every number of unknowns per lane (1025: w
alone fits the lanes).
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, make_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("theta", [1.0, 0.5])
@pytest.mark.parametrize("nz,top", [(5, "dirichlet"), (64, "neumann"), (65, "dirichlet"),
                                    (100, "neumann"), (200, "dirichlet"), (257, "dirichlet"),
                                    (300, "neumann"), (520, "dirichlet"),
                                    (1025, "dirichlet")])
def test_walked_columns_match_single_columns(check, theta, nz, top):
    big = make_plan(_random_case(130, 90, nz, 4, "symmetric", seed=1), nu=1e-2, top=top)
    small = make_plan(_random_case(13, 9, nz, 4, "symmetric", seed=1), nu=1e-2, top=top)
    gen = torch.Generator(device="cuda").manual_seed(nz)
    for comp in "uvw":
        f = torch.randn(big.shapes[comp], dtype=torch.float64, device="cuda", generator=gen)
        before = f.clone()
        big.zsolve(comp, f, 0.02, theta)
        g = torch.empty(small.shapes[comp], dtype=torch.float64, device="cuda")
        ni, nj = g.shape[0], g.shape[1]
        for i0, j0 in [(0, 0), (41, 33), (130 - 13, 90 - 9)]:
            g.copy_(before[i0:i0 + ni, j0:j0 + nj])
            small.zsolve(comp, g, 0.02, theta)
            inner = (slice(1, 14), slice(1, 10))
            check(f"{comp} at {i0},{j0}",
                  torch.equal(g[inner], f[i0 + 1:i0 + 14, j0 + 1:j0 + 10]), "doubles differ")
        check(f"{comp} ghost levels",
              torch.equal(before[..., 0], f[..., 0]) and torch.equal(before[..., -1], f[..., -1]),
              "written")
