"""GPU: the cluster correction of one case at the sizes where its two kernels can go
wrong: clusters of 2, 3, 4, 12 and 18 subdomains (12 to 108 kernel columns: fewer and
more than the lanes of a wave, more than its 16 waves), heat (one column a
subdomain), few and many corner rows (no multiple of 8 or 32).

Bar: within 1e-8 relative of the direct solve (the PCG stops at 1e-11).
"""
import sys

import numpy as np
import pytest

import oracle_lib as O
from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

HEAT = dict(physics=1, length=(1.0, 1.0, 2.0), conductivity=2.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


@pytest.mark.parametrize("heat", [False, True])
@pytest.mark.parametrize("clusters,domains,e", [((2, 1, 1), (2, 1, 1), (2, 2, 2)), ((1, 1, 2), (3, 1, 1), (3, 2, 2)),
                                                ((2, 1, 1), (2, 2, 1), (2, 3, 2)), ((1, 1, 2), (3, 2, 2), (2, 2, 2)),
                                                ((1, 2, 1), (3, 3, 2), (3, 2, 2))])
def test_cluster(heat, clusters, domains, e):
    print("case: cluster of one case", heat, domains, flush=True)
    sys.stdout.flush()
    if heat:
        spec = dict(HEAT, clusters=clusters, domains=domains, elements=e)
    else:
        spec = PB.scaled(PB.GRAVITY, clusters=clusters, domains=domains, elements=e)
    g = core.GridFETI(spec, method="hybrid", precision=1e-11, max_iterations=3000)
    g.setup()
    load = PB.nodal_load_cases(spec, 1, seed=37)[0]
    g.set_nodal_rhs(load)
    g.resolve()
    u = g.nodal_solution()
    g.close()
    direct = O.global_solve_load(spec, load)
    assert np.abs(u - direct).max() < 1e-8 * np.abs(direct).max()
