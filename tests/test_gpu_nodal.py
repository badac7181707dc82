"""GPU: nodal loads and solutions of the structured grid on the device: clusters
of several subdomains (ids not in slab order), uneven slabs, one subdomain, slabs
of one element.

Bars: loads split over 1, 2 or 4 copies and summed again equal the loads bit by bit
(the quarters and their sums are exact), over 8 within two units in the last place
(the sums of 3, 5 and 7 eighths round, by half a unit each); the nodal solution equals the mean of the subdomain
solutions to 1e-15 of its largest value; loads set per subdomain after nodal ones
replace only that subdomain's; a refused load leaves the earlier ones in force.
"""
import numpy as np
import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

CASES = {
    "clusters": dict(PB.GRAVITY, clusters=(2, 1, 2), domains=(2, 2, 1), elements=(2, 3, 2)),
    "uneven": dict(PB.HEAT_UNEVEN_2000, domains=(3, 2, 4), slab_elements=PB.uneven_slabs((3, 2, 4), 3, 1, 5)),
    "one": dict(PB.GRAVITY, clusters=(1, 1, 1), domains=(1, 1, 1), elements=(3, 2, 4)),
    "thin": dict(PB.HEAT_UNEVEN_2000, domains=(4, 1, 2), slab_elements=((1, 1, 2, 1), (3,), (1, 4))),
}


@pytest.mark.parametrize("name", CASES)
def test_nodal_fields(name):
    spec = CASES[name]
    print("case: nodal fields", name, flush=True)
    g = core.GridFETI(spec, preconditioner="dirichlet", precision=1e-11, max_iterations=2000)
    g.setup()
    load = PB.nodal_load_cases(spec, 1, seed=4)[0]
    g.set_nodal_rhs(load)
    copies = np.zeros((len(load), 1))
    for i in range(g.n_sub):
        copies[g.l2g(i)] += 1
    got = g.nodal_load()
    assert np.array_equal(got[copies[:, 0] < 8], load[copies[:, 0] < 8])
    assert np.all(np.abs(got - load) <= 2 * np.spacing(np.abs(load)))
    g.resolve()
    u = g.nodal_solution()
    total = np.zeros_like(u)
    for i in range(g.n_sub):
        nodes = g.l2g(i)
        total[nodes] += g.primal(i, len(nodes) * g.ndof).reshape(len(nodes), g.ndof)
    assert np.abs(u - total / copies).max() <= 1e-15 * np.abs(u).max()
    # a refused load changes nothing
    bad = load.copy()
    bad[-1, 0] = np.inf
    with pytest.raises(RuntimeError, match="non-finite load"):
        g.set_nodal_rhs(bad)
    assert np.array_equal(g.nodal_load(), got)
    # one subdomain's loads replaced on the host: the others keep the nodal ones
    nodes = g.l2g(0)
    f = np.random.default_rng(2).uniform(-1, 1, (len(nodes), g.ndof))
    g.set_rhs(0, f.reshape(-1))
    want = load.copy()
    want[nodes] += f - load[nodes] / copies[nodes]
    assert np.abs(g.nodal_load() - want).max() <= 1e-14
    g.resolve()
    g.set_nodal_rhs(load)
    g.resolve()
    assert np.array_equal(g.nodal_solution(), u)
    g.close()
