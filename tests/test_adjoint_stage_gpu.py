"""The backward stage in one launch (rim groups, band pairs, interior tiles)
against the per-point kernels (`FDM_ADJ_BULK=generic`), at the smallest blocks,
where the band is the whole block, and where a rim group, a workgroup of band
points or a tile is full, one over or nearly empty.

Both sum the same terms in another order: at most 26 terms a point and stage,
each within 2^-53 of its sum, over 25 steps of 5 stages.  Errors add at worst
(26 x 125 x 2^-53 = 3.6e-13 of the terms' size); the bound is 1e-12 of the
largest entry.
"""
import numpy as np
import pytest

import problems
from fdmap_github_amd.adjoint import FaultInversion
from fdmap_github_amd.device import Context

pytestmark = pytest.mark.gpu

DT = 0.5 * 0.025 / np.sqrt(3.464 ** 2 + 6.0 ** 2)
BG = [0.0, 0.0, -120.0, 70.0, -120.0, -120.0]


@pytest.mark.parametrize("nx,nys,nbx,kw", [
    (12, (12, 12), 1, {}), (13, (17, 12), 2, dict(coupling="locked")), (76, (16, 17), 1, dict(law="RAL")),
    (77, (40, 41), 1, dict(law="RSL")), (36, (64, 30), 2, {}),
    (65, (65,), 1, dict(bcs=("absorbing", "free", "rigid", "free")))])
def test_stage_launch_sizes(gpu, monkeypatch, nx, nys, nbx, kw):
    out = []
    for mode in ("tile", "generic"):
        monkeypatch.setenv("FDM_ADJ_BULK", mode)
        prob, F = problems.build(nx=nx, nys=nys, nbx=nbx, seed=nx, warp=0.03, background=BG, perturb=1e-3, **kw)
        ctx = Context(prob)
        ctx.set_fields(F)
        ctx.init_edges(0.0)
        # receivers on an edge, at a corner and inside, one of them twice
        ri = np.array([0, prob.nx - 1, 5, prob.nx // 2, 5], dtype=np.int32)
        rj = np.array([prob.ny // 2, prob.ny - 1, 0, prob.ny // 3, 0], dtype=np.int32)
        inv = FaultInversion(ctx, 0.0, DT, ri, rj, 25, 0)
        rec = inv.run()
        bar = np.random.default_rng(3).standard_normal(rec.shape)
        out.append(inv.adj.backward(bar, fields=True))
        inv.adj.close()
        ctx.close()
    for k in out[0]:
        a, b = np.asarray(out[0][k]), np.asarray(out[1][k])
        assert np.isfinite(b).all()
        assert np.abs(a - b).max(initial=0.0) <= 1e-12 * np.abs(b).max(initial=0.0), (k, np.abs(a - b).max())
