"""The FP32-bulk stage launches of more than 6144 workgroups in a medium or with
dissipation, which run a variant of their own, against the per-point kernel:
the same expressions, so the same bits."""
import numpy as np
import pytest

import problems
from fdmap_github_amd.device import Context

pytestmark = pytest.mark.gpu

DT = 0.5 * 0.025 / np.sqrt(3.464 ** 2 + 6.0 ** 2)


@pytest.mark.parametrize("sbp,kw", [(2, dict(medium=0.2)), (4, dict(medium=0.2)), (4, dict(Cdiss=[200.0, 0.0])),
                                    (4, dict(medium=0.2, Cdiss=200.0)), (6, dict(medium=0.2))])
def test_against_pointwise(gpu, monkeypatch, sbp, kw):
    nx, ny, nb = 1289, 640, {2: 1, 4: 4, 6: 6}[sbp]
    tiles = 2 * -(-(nx - 2 * nb) // 64) * -(-(ny - 2 * nb) // 4)
    assert tiles > 6144
    prob, F = problems.build(nx=nx, nys=(ny, ny), seed=12, warp=0.02, law="RAL", perturb=1e-2, sbp=sbp,
                             background=[0.0, 0.0, -120.0, 70.0, -120.0, -120.0], precision="fp32", **kw)
    out = []
    for env in ({"FDM_BULK": "generic"}, {"FDM_NT_STORE": "0"}, {"FDM_NT_STORE": "1"}):
        for k in ("FDM_BULK", "FDM_NT_STORE", "FDM_BAND_LANES"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        c = Context(prob)
        c.set_fields(F)
        c.init_edges(0.0)
        c.step(0.0, DT, 1, 3)
        out.append(list(c.get_fields()) + list(c.iface_state(0).values()))
        c.close()
    assert all(np.isfinite(a).all() for a in out[0])
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            assert np.array_equal(a, b), np.abs(a - b).max()
