"""Statistics about a provisional mean: fields with means far above their
fluctuations, levels that are exactly uniform, more spectra planes than the
pass marks per level in one word, and a grid large enough for the longest runs.

Moments come from one pass over values less a provisional mean of 64 columns, so
nothing of the size of the mean may be left in their error; a uniform level's
variance must come out as (non-negative) rounding.  Tolerance: the oracle's two
passes see the same doubles, and either side's error is a few ulp of the
fluctuations' moments; 1e-12 of the stresses' scale, as for unit means.
"""

import numpy as np
import pytest

from oracle.turbstats import StatsOracle
from tests.test_stats_hip import TOL, _fields, _rel, _stats

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,mean,extra", [
    ((24, 20, 33), (50.0, -20.0, 3.0), 2), ((5, 3, 66), (50.0, 0.0, 0.0), 2),
    ((18, 14, 40), (1.0, 0.05, 0.0), 34), ((140, 100, 700), (1.0, 0.05, 0.0), 1)])
def test_shifted_moments_match_oracle(check, shape, mean, extra):
    nx, ny, nz = shape
    ts, _ = _stats(nx, ny, nz, planes=[2.0 + 4.0 * q for q in range(extra)])
    planes = [(ts.k_bot, ts.k_top)] + [(p["k_bot"], p["k_top"]) for p in ts.extra_planes]
    orc = StatsOracle(nx, ny, nz, planes=planes)
    u, v, w = _fields(nx, ny, nz, 7, mean)
    for f in (u, v, w):
        f[..., nz // 2] = 0.1  # a uniform level
    orc.accumulate(u.numpy(), v.numpy(), w.numpy())
    ts.accumulate_statistics(u.cuda(), v.cuda(), w.cuda(), 0.05)
    s2 = max(np.max(np.abs(orc.prof[q])) for q in (1, 2, 3, 4))
    for n, q in (("uu", 1), ("vv", 2), ("ww", 3), ("uw", 4)):
        got = getattr(ts, f"{n}_sum").cpu().numpy()
        check(f"{n} within {TOL:g}", _rel(got, orc.prof[q], s2) < TOL,
              f"{_rel(got, orc.prof[q], s2):.1e}")
        if n != "uw":
            check(f"{n} not negative", bool((got >= 0.0).all()), f"{got.min():.1e}")
    s1 = max(np.max(np.abs(orc.prof[q])) for q in (0, 5, 6))
    for n, q in (("U", 0), ("Vm", 5), ("Wm", 6)):
        check(f"{n} within {TOL:g}",
              _rel(getattr(ts, f"{n}_sum").cpu().numpy(), orc.prof[q], s1) < TOL, "means")
    spec = ts._spec.cpu().numpy()
    worst = max(_rel(spec[p], orc.spec[p]) for p in range(len(planes)))
    check(f"{len(planes)} planes' spectra within {TOL:g}", worst < TOL, f"{worst:.1e}")
