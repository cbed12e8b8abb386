"""The antiplane tiles with Ji formed in the kernel and FP32-delta metrics
against the per-point kernel (`FDM_BULK=generic`): the same expressions, so the
same bits, for each operator and option, where the encoding escapes to the
FP64 planes, and with each of the two turned off.
"""
import numpy as np
import pytest

import problems
from fdmap_github_amd import capi
from fdmap_github_amd.device import Context

pytestmark = pytest.mark.gpu

DT = 0.5 * 0.025 / np.sqrt(3.464 ** 2 + 6.0 ** 2)
BG3 = [0.0, 30.0, 40.0]
INPLANE = (-120.0, 0.0, -100.0, -110.0)


def run(monkeypatch, prob, F, env, f32=None):
    for k in ("FDM_BULK", "FDM_JI_CALC", "FDM_METRIC_F32", "FDM_NT_STORE"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    c = Context(prob)
    if f32 is not None:  # raises where the context has no FP32 form
        c._check(c.lib.fdm_tune(c.h, capi.FDM_TUNE_METRIC_F32, f32))
    c.set_fields(F)
    c.init_edges(0.0)
    c.step(0.0, DT, 1, 5)
    out = list(c.get_fields())
    for k in range(len(prob.ifaces)):
        out += list(c.iface_state(k).values())
    c.close()
    return out


@pytest.mark.parametrize("sbp,kw", [(2, {}), (4, {}), (6, {}), (2, dict(medium=0.2)), (6, dict(medium=0.2)),
                                    (4, dict(Cdiss=[200.0, 0.0])), (4, dict(medium=0.2, Cdiss=200.0)),
                                    (4, dict(escape=True)), (6, dict(escape=True))])
def test_variants(gpu, monkeypatch, sbp, kw):
    kw = dict(kw)
    escape = kw.pop("escape", False)
    prob, F = problems.build(nx=81, nys=(33, 42), seed=31, warp=0.0, background=BG3, perturb=1e-2, mode=3,
                             inplane=INPLANE, law="RAL", sbp=sbp, **kw)
    if escape:
        # a few metrics that no FP32 delta holds, Ji still 1/J to the bit
        for m, j, i in (("xq", 20, 40), ("yr", 21, 41), ("xr", 50, 7), ("yq", 70, 80), ("xq", 12, 70)):
            getattr(prob, m)[j, i] += 1e-3 * np.pi
        prob.Ji[:] = 1.0 / (prob.xq * prob.yr - prob.xr * prob.yq)
    ref = run(monkeypatch, prob, F, {"FDM_BULK": "generic"})
    assert all(np.isfinite(a).all() for a in ref)
    for env, f32 in (({}, 1), ({"FDM_NT_STORE": "1"}, 1), ({}, 0), ({"FDM_JI_CALC": "0"}, None)):
        for a, b in zip(run(monkeypatch, prob, F, env, f32), ref):
            assert np.array_equal(a, b), (env, f32, np.abs(a - b).max())
