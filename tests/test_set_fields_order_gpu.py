"""fdm_set_fields follows the steps that are still queued: a context that has
just been stepped and is given new fields goes on as a fresh one does."""
import numpy as np
import pytest

import problems
from fdmap_github_amd.device import Context

pytestmark = pytest.mark.gpu

DT = 0.5 * 0.025 / np.sqrt(3.464 ** 2 + 6.0 ** 2)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_fields_given_while_steps_run(gpu, precision):
    prob, F = problems.build(nx=300, nys=(120,), seed=2, background=[0.0, 0.0, -120.0, 70.0, -120.0, -120.0],
                             perturb=1e-2, precision=precision)
    outs = []
    for before in (0, 400):
        c = Context(prob)
        c.set_fields(F)
        c.init_edges(0.0)
        if before:
            c.step(0.0, DT, 1, before)
            c.set_fields(F)
            c.init_edges(0.0)
        c.step(0.0, DT, 1, 3)
        outs.append(c.get_fields())
        c.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
