"""The step passes of one component per launch against the three in one.

Grids of up to 8192 tiles run the three components in one launch, larger ones
(and any grid while the launch timer is on) a component at a time: other kernels,
which production grids take.  Both must give the same doubles, in every mode,
order and storage, and a grid just past the line must match the direct-load
kernels.
"""

import pytest
import torch

from tests.test_hip_parity import _random_case, cuda, make_plan
from tests.test_tile_boxes_hip import _predictors

pytestmark = pytest.mark.gpu


def _same(check, tag, got, ref):
    for name in ref:
        d = [(a - b).abs() for a, b in zip(got[name][0], ref[name][0])]
        check(f"{tag}: {name}", not any(bool(t.any()) for t in d) and got[name][1] == ref[name][1],
              f"max {max(float(t.max()) for t in d):.1e} ncl {got[name][1]}, {ref[name][1]}")


@pytest.mark.parametrize("storage", [64, 32])
@pytest.mark.parametrize("order", [4, 6])
@pytest.mark.parametrize("shape,cfl", [((20, 18, 33), 1.0), ((21, 19, 22), 4.0),
                                       ((17, 16, 70), 9.0), ((33, 30, 7), 2.0),
                                       ((40, 38, 34), 60.0)])
def test_component_launches_match_merged(check, storage, order, shape, cfl):
    c = _random_case(*shape, order, "symmetric", seed=sum(shape) + order, cfl=cfl)
    plan = make_plan(c, nu=1e-3)
    plan.set_option(plan.OPT_FIELD_STORAGE, storage)
    f = [cuda(a) for a in c["fields"]]
    m = [cuda(a) for a in c["mids"]]
    merged = _predictors(plan, f, m, c["dt"])
    plan.profile(True)
    alone = _predictors(plan, f, m, c["dt"])
    launches = plan.profile_report()
    plan.profile(False)
    check("a launch per component", {"advect_u", "bdf1_v", "bdf2_w"} <= set(launches),
          " ".join(sorted(launches)))
    _same(check, "one component a launch", alone, merged)
    plan.set_option(plan.OPT_BDF2_FUSED, 0)
    split = _predictors(plan, f, m, c["dt"])
    _same(check, "split passes", {"bdf2": split["bdf2"]}, {"bdf2": merged["bdf2"]})


@pytest.mark.parametrize("order", [4, 6])
@pytest.mark.parametrize("shape", [(130, 129, 130), (131, 126, 133)])
def test_grids_past_the_line_match_direct(check, order, shape):
    c = _random_case(*shape, order, "bottom", seed=sum(shape), cfl=2.0)
    plan = make_plan(c, nu=1e-3)
    f = [cuda(a) for a in c["fields"]]
    m = [cuda(a) for a in c["mids"]]
    tiled = _predictors(plan, f, m, c["dt"])
    plan.set_option(plan.OPT_GATHER_TILE, -1)
    _same(check, "tiled == direct", tiled, _predictors(plan, f, m, c["dt"]))
