"""GPU: the row norms of S_D and F_i (the scale of the SYMV's fixed-point sums; a norm
that is too small wraps them): one block of 64 rows, several with a ragged last one,
many small subdomains, and many of more than 256 rows.

Bar: the KKT residuals of a solve, which come from K u - f and not from F_i, below
1e-9: rounding of the local solves (about 1e-16 times their condition, below 1e5).
"""
import sys

import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


def heat(subs, e):
    return dict(physics=1, clusters=subs, domains=(1, 1, 1), elements=e, length=(1.0, 1.0, 1.0), conductivity=2.0,
                heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


@pytest.mark.parametrize("spec", [heat((1, 1, 2), (3, 3, 3)), PB.scaled(PB.GRAVITY, clusters=(2, 1, 1),
                                                                       domains=(1, 1, 1), elements=(6, 5, 4)),
                                  heat((11, 10, 10), (3, 3, 3)), heat((8, 8, 9), (9, 9, 8))])
def test_norms(spec):
    print("case: row norms", spec["clusters"], spec["elements"], flush=True)
    sys.stdout.flush()
    g = core.GridFETI(spec, precision=1e-10, max_iterations=2000)
    g.setup()
    s = g.solve()
    g.close()
    print("  kkt", s["kkt_primal"], s["kkt_dual"], flush=True)
    assert s["kkt_primal"] < 1e-9 and s["kkt_dual"] < 1e-9
