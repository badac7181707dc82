"""GPU: set-ups whose assembly workspace holds the largest subdomain only without the
padding of its columns: four waves a tile (few subdomains) and one wave a tile (a large
subdomain whose workspace holds about a hundred small ones).

The smallest budget that is accepted is the unpadded workspace of the largest subdomain;
its numbers of interior and interface DOFs are no multiples of 16, so the padded one is
larger by more than the budget's margin.  S_D and F_i against numpy as S = K_bb - K_bi K_ii^-1 K_ib and
F = (S + rho Q Q^T)^-1, rho = max diag S, Q the orthonormal kernel on the interface, or, for
the largest, against the padded set-up; both to 1e-9 of the largest entry (n eps cond with
n <= 1e4, cond <= 1e3; solutions to 1e-8, the stop test is 1e-11).
"""
import numpy as np
import pytest

from espreso_amd import core

pytestmark = pytest.mark.gpu
MARGIN = 1.0 + 1e-4


def solver(spec, budget_gb=0.0):
    return core.GridFETI(spec, preconditioner="dirichlet", precision=1e-11, max_iterations=2000,
                         memory_budget_gb=budget_gb)


def accepted(spec, budget_gb):
    with solver(spec, budget_gb) as g:
        try:
            g.setup()
        except RuntimeError as e:
            assert "assembly workspace exceeds" in str(e)
            return False
        return True


def smallest_budget(spec):
    """GB, to the margin."""
    b = 1e-6
    while not accepted(spec, b):
        b *= 2.0
    a = 0.5 * b
    while b > a * (0.5 * (1.0 + MARGIN)):
        c = 0.5 * (a + b)
        if accepted(spec, c):
            b = c
        else:
            a = c
    return b


def reference(spec, g, i):
    d = core.grid_export(spec, i)
    K = np.zeros((d["n"], d["n"]))
    for r in range(d["n"]):
        q = slice(d["rowptr"][r], d["rowptr"][r + 1])
        K[r, d["colidx"][q]] = d["vals"][q]
    b = g.boundary(i)
    o = np.setdiff1d(np.arange(d["n"]), b)
    S = K[np.ix_(b, b)] - K[np.ix_(b, o)] @ np.linalg.solve(K[np.ix_(o, o)], K[np.ix_(o, b)])
    Q, _ = np.linalg.qr(d["R"][b])
    return np.linalg.inv(S + np.diag(S).max() * Q @ Q.T), S, len(o)


def heat(domains, elements, slabs=None):
    spec = dict(physics=1, clusters=(1, 1, 1), domains=domains, elements=elements, length=(1.0, 1.0, 1.0),
                conductivity=1.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))
    return dict(spec, slab_elements=slabs) if slabs else spec


def elasticity(domains, elements, slabs=None):
    spec = dict(physics=0, clusters=(1, 1, 1), domains=domains, elements=elements, length=(1.0, 1.0, 1.0), young=1.0,
                poisson=0.3, accel=(0.0, 0.0, -1.0), density=1.0, fixed=(0, 0, 0, 0, 7, 0))
    return dict(spec, slab_elements=slabs) if slabs else spec


# 14^3 elements in the corner and 3^3 elsewhere: waves of two layers, about 100 subdomains, of which the
# largest has 27 interface tiles, pass the numbers of tiles at which the one-wave kernels take over
UNEVEN = tuple((14,) + (3,) * 6 for _ in range(3))


@pytest.mark.parametrize("spec,checked", [
    (heat((1, 1, 2), (2, 4, 3)), (0, 1)), (heat((2, 2, 2), (4, 5, 6)), (0, 3, 7)),
    (elasticity((2, 2, 2), (3, 5, 4)), (0, 7)), (elasticity((7, 7, 7), (3, 3, 3), UNEVEN), (8, 49 + 7, 171, 342))])
def test_unpadded_workspace(spec, checked):
    print("case: small workspace", spec["physics"], spec["domains"], spec["elements"], flush=True)
    budget = smallest_budget(spec)
    with solver(spec) as padded, solver(spec, budget * MARGIN) as g:
        padded.setup()
        padded.solve()
        g.setup()
        g.solve()
        print(f"  {budget * 1e3:.4f} MB", flush=True)
        for i in checked:
            F, S, ni = reference(spec, g, i)
            for which, want in ((0, F), (1, S)):
                err = np.abs(g.dense(i, which) - want).max() / np.abs(want).max()
                print(f"  subdomain {i}: interior {ni}, interface {len(S)}, {'S_D' if which else 'F'} {err:.1e}", flush=True)
                assert err < 1e-9
        for which in (0, 1):
            want = padded.dense(0, which)
            assert np.abs(g.dense(0, which) - want).max() < 1e-9 * np.abs(want).max()
        u = padded.nodal_solution()
        assert np.abs(g.nodal_solution() - u).max() < 1e-8 * np.abs(u).max()
