"""GPU: the assembly's 64 x 64 diagonal tiles (Cholesky factor and inverse) at
their edges: interiors and interfaces of less than a 16-column block, of one
block more or less than a tile, of a whole number of tiles and of several.

S_D and F_i of single subdomains of a 1 x 1 x 2 heat or elasticity row against
numpy: S = K_bb - K_bi K_ii^-1 K_ib from the exported K_i, and F from
F = (S + rho Q Q^T)^-1 with Q the orthonormal kernel on the interface and rho =
max diag S.  Bar: 1e-9 relative to the largest entry (n eps cond with n <= 1e3,
cond <= 1e4 leaves a margin of ten); a K_i that is not positive definite on the
interior is reported with its first failing column.
"""
import numpy as np
import pytest

from espreso_amd import core

pytestmark = pytest.mark.gpu


def row(physics, ex, ey, ez):
    spec = dict(physics=physics, clusters=(1, 1, 1), domains=(1, 1, 2), elements=(ex, ey, ez), length=(1.0, 1.0, 2.0))
    if physics == 0:
        spec.update(young=1.0, poisson=0.3, accel=(0.0, 0.0, -1.0), density=1.0, fixed=(0, 0, 0, 0, 7, 0))
    else:
        spec.update(conductivity=1.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))
    return spec


# interior and interface sizes of the second subdomain (interface z = 0 only):
# heat (ex+1)(ey+1) interface, (ex+1)(ey+1)ez interior DOFs; three times that in elasticity
@pytest.mark.parametrize("physics,ex,ey,ez", [
    (1, 1, 1, 1), (1, 2, 4, 1), (1, 3, 3, 1), (1, 4, 2, 1), (1, 7, 7, 1), (1, 4, 12, 1), (1, 8, 8, 2), (1, 15, 7, 3),
    (0, 1, 1, 1), (0, 2, 6, 1), (0, 4, 4, 2), (0, 6, 8, 3)])
def test_tiles(physics, ex, ey, ez):
    spec = row(physics, ex, ey, ez)
    print("case: tiles", physics, ex, ey, ez, flush=True)
    g = core.GridFETI(spec, preconditioner="dirichlet")
    g.setup()
    for i in range(2):
        d = core.grid_export(spec, i)
        K = np.zeros((d["n"], d["n"]))
        for r in range(d["n"]):
            q = slice(d["rowptr"][r], d["rowptr"][r + 1])
            K[r, d["colidx"][q]] = d["vals"][q]
        b = g.boundary(i)
        o = np.setdiff1d(np.arange(d["n"]), b)
        S = K[np.ix_(b, b)]
        if len(o):
            S = S - K[np.ix_(b, o)] @ np.linalg.solve(K[np.ix_(o, o)], K[np.ix_(o, b)])
        Q, _ = np.linalg.qr(d["R"][b])
        F = np.linalg.inv(S + np.diag(S).max() * Q @ Q.T)
        for which, want in ((1, S), (0, F)):
            got = g.dense(i, which)
            err = np.abs(got - want).max() / np.abs(want).max()
            print(f"  subdomain {i}: interior {len(o)}, interface {len(b)}, {'S_D' if which else 'F'} {err:.1e}", flush=True)
            assert err < 1e-9
    g.close()


@pytest.mark.parametrize("col", [0, 15, 16, 70])
def test_breakdown_column(col):
    spec = row(1, 8, 8, 2)
    print("case: breakdown", col, flush=True)
    g = core.GridFETI(spec, preconditioner="dirichlet")
    g.setup()
    d = core.grid_export(spec, 1)
    b = g.boundary(1)
    o = np.setdiff1d(np.arange(d["n"]), b)
    v = d["vals"].copy()
    r = o[col]
    for q in range(d["rowptr"][r], d["rowptr"][r + 1]):
        if d["colidx"][q] == r:
            v[q] = -1.0
    g.update_values(1, v)
    with pytest.raises(RuntimeError, match=f"subdomain 1 at column {col + 1}$"):
        g.setup()
    g.close()


# wave tiles take over from four waves per tile at 2048 substitution, 1024 panel and
# 8192 SYRK tiles in a launch: 512 to 1000 subdomains whose interiors and interfaces
# end just before, on and after a tile, checked in the first, an inner and the last one
@pytest.mark.parametrize("physics,domains,elements", [
    (1, (10, 10, 10), (6, 6, 6)), (1, (8, 8, 8), (7, 6, 5)), (0, (8, 8, 8), (3, 4, 4)), (0, (8, 8, 8), (5, 5, 4)),
    (0, (6, 6, 6), (7, 7, 7))])
def test_wave_tiles(physics, domains, elements):
    spec = dict(row(physics, *elements), domains=domains, length=(1.0, 1.0, 1.0))
    print("case: wave tiles", physics, domains, elements, flush=True)
    n = int(np.prod(domains))
    g = core.GridFETI(spec, preconditioner="dirichlet")
    g.setup()
    for i in (0, n // 2 + domains[0] // 2, n - 1):
        d = core.grid_export(spec, i)
        K = np.zeros((d["n"], d["n"]))
        for r in range(d["n"]):
            q = slice(d["rowptr"][r], d["rowptr"][r + 1])
            K[r, d["colidx"][q]] = d["vals"][q]
        b = g.boundary(i)
        o = np.setdiff1d(np.arange(d["n"]), b)
        S = K[np.ix_(b, b)] - K[np.ix_(b, o)] @ np.linalg.solve(K[np.ix_(o, o)], K[np.ix_(o, b)])
        Q, _ = np.linalg.qr(d["R"][b])
        F = np.linalg.inv(S + np.diag(S).max() * Q @ Q.T)
        for which, want in ((1, S), (0, F)):
            err = np.abs(g.dense(i, which) - want).max() / np.abs(want).max()
            print(f"  subdomain {i}: interior {len(o)}, interface {len(b)}, {'S_D' if which else 'F'} {err:.1e}", flush=True)
            assert err < 1e-9
    g.close()
