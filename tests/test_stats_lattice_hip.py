"""Statistics of fields that the provisional mean's 8 x 8 columns see one-sidedly.

The moments are sums about a mean of 64 columns on a regular lattice.  With m the
error of that mean and s2 the variance, the final subtraction takes m^2 from
s2 + m^2, and so loses a factor of up to 1 + 2 m^2 / s2 to rounding.  A pattern in
phase with the lattice has m^2 = 4 s2; values on its columns alone have m^2 near
N / 64 s2 for N columns, the worst there is (Cauchy-Schwarz).

Tolerance: a sum's terms pass through fewer than 200 additions on either side,
so 200 ulp of the sum of squares about the provisional mean, which is
1 + 2 m^2 / s2 of the variance; 200 ulp of the provisional mean's size for the
means; TOL for the spectra, whose transform's rounding is that of the plane's
norm.
"""

import math

import numpy as np
import pytest
import torch

from oracle.turbstats import StatsOracle
from tests.test_stats_hip import TOL, _rel, _stats

pytestmark = pytest.mark.gpu

SIDE = 8


def _columns(n):
    return [c * n // SIDE + 1 for c in range(SIDE)]


def _pattern(kind, shape, nx, ny):
    i, j = np.arange(shape[0])[:, None], np.arange(shape[1])[None, :]
    if kind == "phase":
        return np.cos(2 * math.pi * SIDE * (i - 1) / nx) * np.cos(2 * math.pi * SIDE * (j - 1) / ny)
    return (np.isin(i, _columns(nx)) & np.isin(j, _columns(ny))).astype(float)


@pytest.mark.parametrize("kind", ["phase", "columns"])
@pytest.mark.parametrize("nx,ny,nz", [(64, 48, 20), (160, 128, 33)])
def test_lattice_fields_match_oracle(check, kind, nx, ny, nz):
    ts, _ = _stats(nx, ny, nz, planes=[40.0])
    planes = [(ts.k_bot, ts.k_top)] + [(p["k_bot"], p["k_top"]) for p in ts.extra_planes]
    orc = StatsOracle(nx, ny, nz, planes=planes)
    gen = torch.Generator().manual_seed(nx)
    f, worst, size = [], 0.0, 0.0
    for amp, s in zip((1.0, 0.7, 0.4), ((nx + 1, ny + 2, nz + 2), (nx + 2, ny + 1, nz + 2),
                                        (nx + 2, ny + 2, nz + 1))):
        a = 1e-3 * torch.randn(s, generator=gen, dtype=torch.float64)
        a += torch.from_numpy(amp * _pattern(kind, s, nx, ny))[:, :, None]
        nodes = a.numpy()[1:nx + 1, 1:ny + 1]
        lattice = nodes[np.ix_([c - 1 for c in _columns(nx)], [c - 1 for c in _columns(ny)])]
        m = lattice.mean((0, 1)) - nodes.mean((0, 1))
        worst = max(worst, float((m * m / nodes.var((0, 1))).max()))
        size = max(size, float(np.abs(lattice.mean((0, 1))).max()))
        f.append(a)
    check("the lattice misses the mean", worst > (3.0 if kind == "phase" else 0.5 * nx * ny / 64),
          f"m^2 / s2 = {worst:.1f}")
    orc.accumulate(*(a.numpy() for a in f))
    ts.accumulate_statistics(*(a.cuda() for a in f), 0.05)
    ulp = 200 * np.finfo(float).eps
    s2 = max(np.max(np.abs(orc.prof[q])) for q in (1, 2, 3, 4))
    for n, q in (("uu", 1), ("vv", 2), ("ww", 3), ("uw", 4)):
        e = _rel(getattr(ts, f"{n}_sum").cpu().numpy(), orc.prof[q], s2)
        check(f"{n}", e < ulp * (1 + 2 * worst), f"{e:.1e} of {ulp * (1 + 2 * worst):.1e}")
    s1 = max(np.max(np.abs(orc.prof[q])) for q in (0, 5, 6))
    for n, q in (("U", 0), ("Vm", 5), ("Wm", 6)):
        e = _rel(getattr(ts, f"{n}_sum").cpu().numpy(), orc.prof[q], s1)
        check(f"{n}", e * s1 < 2 * ulp * size, f"{e * s1:.1e} of {2 * ulp * size:.1e}")
    spec = ts._spec.cpu().numpy()
    e = max(_rel(spec[p], orc.spec[p]) for p in range(len(planes)))
    check("spectra", e < TOL, f"{e:.1e}")
