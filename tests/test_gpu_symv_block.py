"""GPU: the block SYMV where its split can go wrong: one item of fewer strips than
waves (26 and 42 boundary DOFs), an item whose last strip is ragged (78: 5 strips),
items of 8 + 3 strips (168), 8 + 8 + 3 (294), 8 + 2 with a tenth of 2 rows (146),
and 3, 15 and 16 cases (idle lanes, the full MFMA width).

Bar: each case within 1e-8 relative of the direct solve (the PCG stops at 1e-11).
"""
import sys

import numpy as np
import pytest

import oracle_lib as O
from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


def heat(e):
    return dict(physics=1, clusters=(1, 1, 2), domains=(1, 1, 1), elements=e, length=(1.0, 1.0, 2.0),
                conductivity=2.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


def elasticity(e):
    return PB.scaled(PB.GRAVITY, clusters=(2, 1, 1), domains=(1, 1, 1), elements=e)


@pytest.mark.parametrize("spec,m", [(heat((2, 2, 2)), 26), (heat((2, 2, 4)), 42), (elasticity((2, 2, 2)), 78),
                                    (heat((4, 4, 7)), 146), (elasticity((3, 3, 3)), 168),
                                    (elasticity((4, 4, 4)), 294)])
@pytest.mark.parametrize("ncases", [3, 15, 16])
def test_block_items(spec, m, ncases):
    print("case: block items", m, ncases, flush=True)
    sys.stdout.flush()
    e = spec["elements"]
    nodes = (e[0] + 1) * (e[1] + 1) * (e[2] + 1) - (e[0] - 1) * (e[1] - 1) * (e[2] - 1)
    assert nodes * (1 if spec["physics"] == 1 else 3) == m
    g = core.GridFETI(spec, precision=1e-11, max_iterations=2000)
    g.setup()
    loads = PB.nodal_load_cases(spec, ncases, seed=5)
    ub, _, _ = g.resolve_block_nodal(loads)
    g.close()
    for q in range(ncases):
        direct = O.global_solve_load(spec, loads[q])
        assert np.abs(ub[q] - direct).max() < 1e-8 * np.abs(direct).max(), q
