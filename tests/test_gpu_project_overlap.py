"""GPU: allocation-free projections of several instances in flight at once, on their own
streams and on a stream of the caller, equal the projections made one by one bit by bit."""
import numpy as np
import pytest
import torch

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

SPECS = [dict(PB.GRAVITY, clusters=(4, 4, 4), domains=(1, 1, 1), elements=(3, 3, 3)),
         dict(PB.GRAVITY, clusters=(6, 5, 4), domains=(1, 1, 1), elements=(3, 2, 2)),
         dict(PB.GRAVITY, clusters=(2, 2, 2), domains=(2, 2, 2), elements=(3, 3, 3), method="hybrid")]


def test_overlapping_projections():
    print("case: overlapping projections", flush=True)
    mine = torch.cuda.Stream()
    solvers = []
    for spec in SPECS:
        spec = dict(spec)
        g = core.GridFETI(spec, method=spec.pop("method", "total"), preconditioner="lumped")
        g.setup()
        solvers.append(g)
    rng = np.random.default_rng(41)
    x = [rng.standard_normal((40, g.n_lambda)) for g in solvers]
    dx = [torch.from_numpy(v).cuda() for v in x]
    dy = [torch.full_like(v, float("nan")) for v in dx]
    torch.cuda.synchronize()
    for i in range(40):
        for k, g in enumerate(solvers):
            g.project_device(dx[k][i].data_ptr(), dy[k][i].data_ptr(), mine.cuda_stream if k == 1 else None)
    torch.cuda.synchronize()
    for k, g in enumerate(solvers):
        want = np.stack([g.project(v) for v in x[k]])
        assert np.array_equal(dy[k].cpu().numpy(), want), k
        g.close()
