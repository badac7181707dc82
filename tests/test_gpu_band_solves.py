"""GPU: the interior band solves at the sizes where their tiles can go wrong: one
interior DOF, 63 (7 x 3 x 3), 64, 80 and 81 (a second block of 16 and 17), 2187 with
a band past 16 tiles, many subdomains, and 1,
2, 5, 16 and 17 cases (one case, idle lanes, the full width, two chunks).

Bar: each case within 1e-8 relative of the direct solve (the PCG stops at 1e-11).
"""
import sys

import numpy as np
import pytest

import oracle_lib as O
from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


def heat(e, clusters=(1, 1, 2)):
    return dict(physics=1, clusters=clusters, domains=(1, 1, 1), elements=e, length=(1.0, 1.0, 2.0),
                conductivity=2.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


def elasticity(e):
    return PB.scaled(PB.GRAVITY, clusters=(2, 1, 1), domains=(1, 1, 1), elements=e)


@pytest.mark.parametrize("spec,ni,ncases", [
    (heat((2, 2, 2)), 1, 1), (heat((2, 2, 2)), 1, 17), (heat((8, 4, 4)), 63, 2), (heat((5, 5, 5)), 64, 5),
    (heat((5, 5, 6)), 80, 16), (elasticity((4, 4, 4)), 81, 1), (elasticity((4, 4, 4)), 81, 17),
    (elasticity((10, 10, 10)), 2187, 1), (elasticity((10, 10, 10)), 2187, 5),
    (heat((5, 5, 5), (7, 7, 6)), 64, 1), (heat((6, 5, 5), (7, 7, 6)), 80, 3)])
def test_band(spec, ni, ncases):
    print("case: band", ni, ncases, flush=True)
    sys.stdout.flush()
    e = spec["elements"]
    assert (e[0] - 1) * (e[1] - 1) * (e[2] - 1) * (1 if spec["physics"] == 1 else 3) == ni
    g = core.GridFETI(spec, precision=1e-11, max_iterations=2000)
    g.setup()
    loads = PB.nodal_load_cases(spec, ncases, seed=11)
    direct = [O.global_solve_load(spec, f) for f in loads]
    for q in range(min(ncases, 2)):
        g.set_nodal_rhs(loads[q])
        g.resolve()
        assert np.abs(g.nodal_solution() - direct[q]).max() < 1e-8 * np.abs(direct[q]).max(), q
    ub, _, _ = g.resolve_block_nodal(loads)
    g.close()
    for q in range(ncases):
        assert np.abs(ub[q] - direct[q]).max() < 1e-8 * np.abs(direct[q]).max(), q
