"""GPU: the PCG kernels on interleaved load cases at the sizes where their line
layout can go wrong: 1, 2, 7 and 16 cases (one line per thread, lines that do
and do not divide the workgroup), coarse spaces that are no multiple of the 16
MFMA rows (3 elasticity subdomains: 18, 5 heat subdomains: 5), one workgroup and
several, every preconditioner, with and without clusters.

Bars: each case within 1e-8 relative of the direct solve, solved in the block
and alone (the PCG stops at 1e-11); the projector idempotent to 1e-12.
"""
import sys

import numpy as np
import pytest

import oracle_lib as O
from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

ROW = PB.scaled(PB.GRAVITY, clusters=(3, 1, 1), domains=(1, 1, 1), elements=(2, 3, 2))
HEAT = dict(physics=1, clusters=(1, 1, 5), domains=(1, 1, 1), elements=(3, 2, 4), length=(1.0, 1.0, 2.0),
            conductivity=2.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))
HYBRID = PB.scaled(PB.GRAVITY, clusters=(2, 1, 1), domains=(2, 1, 2), elements=(3, 3, 2))


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("spec,method,prec,ncases", [
    (ROW, "total", "dirichlet", 1), (ROW, "total", "lumped", 7), (HEAT, "total", "dirichlet", 16),
    (HEAT, "total", "weight", 2), (ROW, "total", "super_dirichlet", 16), (HEAT, "total", "none", 7),
    (HYBRID, "hybrid", "dirichlet", 7), (HYBRID, "hybrid", "super_dirichlet", 2), (HYBRID, "hybrid", "lumped", 16)])
def test_lines(spec, method, prec, ncases):
    print("case: lines", spec["physics"], method, prec, ncases, flush=True)
    sys.stdout.flush()
    g = core.GridFETI(spec, method=method, preconditioner=prec, precision=1e-11, max_iterations=3000)
    g.setup()
    x = np.random.default_rng(3).standard_normal(g.n_lambda)
    px = g.project(x)
    assert rel(g.project(px), px) < 1e-12
    loads = PB.nodal_load_cases(spec, ncases, seed=17)
    ub, itb, nrm = g.resolve_block_nodal(loads)
    for q in range(ncases):
        g.set_nodal_rhs(loads[q])
        st = g.resolve()
        alone = g.nodal_solution()
        direct = O.global_solve_load(spec, loads[q])
        print(f"  case {q}: iterations {itb[q]} / {st['iterations']}, vs direct {rel(ub[q], direct):.2e}, vs alone "
              f"{rel(ub[q], alone):.2e}", flush=True)
        assert rel(ub[q], direct) < 1e-8 and rel(alone, direct) < 1e-8
    g.close()
