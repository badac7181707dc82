"""GPU: the work items of the SYMV at the sizes where the rule for small operators
changes: subdomains smaller than the smallest item (1 item), cut at that size (8
subdomains of 654 boundary DOFs), cut for the number of workgroups (27 of 1158), in
every storage precision, against one item per subdomain.

Bar: both are sums of at most m products in another order, in the accumulation
type (FP64, FP32 for FP32 and BF16 storage), so they differ by at most
2 m eps sum_j |F_ij x_j|; for a random x that sum is about sqrt(m) |y_i|.
"""
import sys

import numpy as np
import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sub,e,m", [((2, 1, 1), 2, 78), ((2, 2, 2), 6, 654), ((3, 3, 3), 8, 1158)])
@pytest.mark.parametrize("sc,eps", [("fp64", 2.0**-53), ("fp32", 2.0**-24), ("bf16", 2.0**-24)])
def test_items(monkeypatch, sub, e, m, sc, eps):
    print("case: items", sub, e, sc, flush=True)
    sys.stdout.flush()
    assert 3 * ((e + 1)**3 - (e - 1)**3) == m
    spec = PB.scaled(PB.GRAVITY, clusters=sub, domains=(1, 1, 1), elements=(e, e, e))
    y = []
    for item in (None, "1310720"):
        if item:
            monkeypatch.setenv("ESPRESO_SYMV_ITEM", item)
        g = core.GridFETI(spec, sc_precision=sc)
        g.setup()
        x = np.random.default_rng(23).standard_normal(g.n_lambda)
        y.append(g.apply_F(x))
        assert np.array_equal(y[-1], g.apply_F(x))
        g.close()
    assert np.abs(y[0] - y[1]).max() < 2 * m**1.5 * eps * np.abs(y[1]).max()
