"""GPU: the row norms of F_i and S_D against numpy, at interfaces of less than a 64-row
block, of whole blocks and one more, and of several.

The SYMV's sums are multiples of 2^-k with k = 60 - floor(log2(2 ||A||_inf max|x|)), exactly
as long as they stay below 2^53 of these units.  The rows of held DOFs have one entry each, so
for x on one of them the smallest bit among the outputs on the held rows of its subdomain is
2^-k (one work item per subdomain; hundreds of sums, of which some are odd multiples).  The
scale c of x at which k steps gives the norm; 14 bisections of [1, 2) know it to 1.3e-4.
"""
import numpy as np
import pytest

from espreso_amd import core

pytestmark = pytest.mark.gpu


def lowest_bit(y):
    """Exponent of the lowest bit set in any of the values."""
    m, e = np.frexp(y[y != 0.0])
    m = np.abs(np.ldexp(m, 53)).astype(np.int64)
    return int((np.log2(m & -m).astype(int) + e - 53).min())


def norm_seen(apply, x, rows):
    low = lowest_bit(apply(x)[rows])
    a, b = 1.0, 2.0  # low at a, low + 1 at b
    for _ in range(14):
        c = 0.5 * (a + b)
        if lowest_bit(apply(c * x)[rows]) > low:
            b = c
        else:
            a = c
    # 2 norm b = 2^(60 - k + 1) with -k = low
    return 2.0 ** (60 + low) / b


# interface rows (the cut and the held face x = 0): heat 63, 64, 65 and 260, elasticity 120 and 510
@pytest.mark.parametrize("physics,ex,ey,ez", [(1, 4, 6, 4), (1, 8, 3, 7), (1, 6, 4, 6), (1, 10, 12, 9), (0, 4, 4, 3),
                                              (0, 6, 9, 10)])
def test_norms(monkeypatch, physics, ex, ey, ez):
    monkeypatch.setenv("ESPRESO_SYMV_ITEM", str(1 << 30))
    held = 7 if physics == 0 else 1
    spec = dict(physics=physics, clusters=(1, 1, 1), domains=(1, 1, 2), elements=(ex, ey, ez), length=(1.0, 1.0, 2.0),
                fixed=(held, 0, 0, 0, 0, 0))
    if physics == 0:
        spec.update(young=1.0, poisson=0.3, accel=(0.0, 0.0, -1.0), density=1.0)
    else:
        spec.update(conductivity=1.0, heat_source=1.0)
    with core.GridFETI(spec, preconditioner="dirichlet", scaling=0) as g:
        g.setup()
        exports = [core.grid_export(spec, i, scaling=0) for i in range(2)]
        count = np.bincount(np.concatenate([d["lam"] for d in exports]), minlength=g.n_lambda)
        for i, d in enumerate(exports):
            rows = d["lam"][(count[d["lam"]] == 1) & (d["scale"] == 1.0)]
            x = np.zeros(g.n_lambda)
            x[rows[len(rows) // 2]] = 1.0
            for which, apply in ((0, g.apply_F), (1, g.apply_prec)):
                want = np.abs(g.dense(i, which)).sum(1).max()
                got = norm_seen(apply, x, rows)
                print(f"case: norms {physics} {ex} {ey} {ez}, subdomain {i} of {len(g.boundary(i))} rows, "
                      f"{'S_D' if which else 'F'}: {got:.6e} {want:.6e}", flush=True)
                assert abs(got / want - 1.0) < 2e-4
