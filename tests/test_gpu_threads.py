"""GPU: instances in several threads, each set up, solved, re-solved (one load and a block, which
capture graphs) and closed while the others do the same, give the bits of the same calls
made in one thread."""
import threading

import numpy as np
import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

CASES = [(PB.TFETI_64x5, {}), (dict(PB.GRAVITY, clusters=(2, 2, 2), domains=(2, 2, 2), elements=(4, 3, 4)),
                               dict(method="hybrid")),
         (dict(PB.GRAVITY, clusters=(3, 3, 3), domains=(1, 1, 1), elements=(4, 4, 3)),
          dict(sc_precision="fp32", sd_precision="bf16"))]


def work(case, out):
    spec, opts = case
    for rep in range(3):
        with core.GridFETI(spec, preconditioner="dirichlet", precision=1e-9, max_iterations=1000, **opts) as g:
            g.setup()
            g.solve()
            out.append(g.nodal_solution())
            loads = PB.nodal_load_cases(spec, 3, seed=rep)
            g.set_nodal_rhs(loads[0])
            g.resolve()
            out.append(g.nodal_solution())
            out.append(np.array(g.resolve_block_nodal(loads)[0]))
            x = np.random.default_rng(rep).standard_normal(g.n_lambda)
            out += [g.apply_F(x), g.apply_prec(x), g.project(x)]


def test_threads():
    print("case: instances in threads", flush=True)
    alone = [[] for _ in CASES]
    for case, out in zip(CASES, alone):
        work(case, out)
    for _ in range(3):
        got, errors = [[] for _ in CASES], []

        def run(k):
            try:
                work(CASES[k], got[k])
            except Exception as e:  # reported by the test's own thread
                errors.append(e)

        threads = [threading.Thread(target=run, args=(k,)) for k in range(len(CASES))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors
        for a, b in zip(alone, got):
            assert len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))
