"""GPU: the band copy of the K_ii factor where the band reaches past the factor's band
tiles: interior planes of exactly 64 DOFs (8 x 8 heat nodes: one tile of band by tiles,
73 columns of band by DOFs), whose columns' last rows lie in a tile that the
factorisation neither writes nor reads.  The workspace holds an earlier instance's values
by then, so the first solve of a process says nothing.

Bar: the KKT residuals of the solve and of a re-solve below 1e-9 (rounding of the local
solves), the solution of both the same to 1e-9.
"""
import sys

import numpy as np
import pytest

from espreso_amd import core

pytestmark = pytest.mark.gpu


def heat(subs, e):
    return dict(physics=1, clusters=subs, domains=(1, 1, 1), elements=e, length=(1.0, 1.0, 1.0), conductivity=2.0,
                heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


@pytest.mark.parametrize("subs", [(3, 3, 3), (4, 4, 5)])
def test_planes(subs):
    print("case: band tiles", subs, flush=True)
    sys.stdout.flush()
    for spec in (heat((4, 4, 4), (7, 6, 8)), heat(subs, (9, 9, 8))):
        g = core.GridFETI(spec, precision=1e-9, max_iterations=500)
        g.setup()
        s = g.solve()
        u = g.nodal_solution()
        assert s["kkt_primal"] < 1e-9 and s["kkt_dual"] < 1e-9
        g.set_nodal_rhs(g.nodal_load())
        s = g.resolve()
        assert s["kkt_primal"] < 1e-9
        assert np.abs(g.nodal_solution() - u).max() < 1e-9 * np.abs(u).max()
        g.close()
