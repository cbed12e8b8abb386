"""fdm_profile_read counts stages: one entry a stage whatever the number of
launches behind it, and every grid point in each."""
import numpy as np
import pytest

import problems
from fdmap_github_amd.device import Context

pytestmark = pytest.mark.gpu

DT = 0.5 * 0.025 / np.sqrt(3.464 ** 2 + 6.0 ** 2)
LAYER = dict(x=True, y=True, sigma=15.0, kappa=0.2)


@pytest.mark.parametrize("bulk", ["tile", "generic"])
@pytest.mark.parametrize("kw", [{}, dict(pml=LAYER), dict(pml=[LAYER, None]), dict(pml=[None, LAYER])],
                         ids=["none", "all", "first", "second"])
def test_one_entry_a_stage(gpu, monkeypatch, kw, bulk):
    monkeypatch.setenv("FDM_BULK", bulk)
    prob, F = problems.build(nx=90, nys=(40, 36), seed=6, perturb=1e-3, law="RFL",
                             background=[0.0, 0.0, -120.0, 70.0, -120.0, -120.0], **kw)
    c = Context(prob)
    c.set_fields(F)
    c.init_edges(0.0)
    c.profile_enable(True)
    c.step(0.0, DT, 1, 6)
    c.stage1(0.0, DT, 7)
    p = c.profile_read()
    stages = 6 * 5 + 1
    assert p["bulk_launches"] == stages and p["bulk_points"] == prob.nx * prob.ny and p["bulk_ms"] > 0.0
    assert p["edge_launches"] == (stages if bulk == "generic" else 0)
    assert p["band_launches"] == 0 and p["band_ms"] == 0.0
    c.close()
