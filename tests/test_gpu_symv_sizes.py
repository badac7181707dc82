"""GPU: the SYMV work items that run are the ones that are reported, and an operator
takes no size that was timed on another one.

A work list decides the grouping of the sums of F x, so two instances of one problem
give equal bits exactly when they run the same list: a size fixed by
ESPRESO_SYMV_ITEM runs as it is, and the tuned and the default size have to give
its bits (sizes under 98304 are reported as 98304).
"""
import numpy as np
import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu

FINE = (98304, 49152, 32768, 16384)


def spec_of(sub, elements):
    return PB.scaled(PB.GRAVITY, clusters=sub, domains=(1, 1, 1), elements=elements)


def apply_F(spec):
    with core.GridFETI(spec, preconditioner="lumped") as g:
        g.setup()
        return g.apply_F(np.random.default_rng(29).standard_normal(g.n_lambda)), g.symv_items()[0]


# one subdomain or a few (11 items of 320 K each at 12^3), where the items were cut for the number of
# workgroups; 512 of 5^3: more elements than 1024 items of 48 K hold
@pytest.mark.parametrize("sub,e", [((1, 1, 1), 5), ((2, 2, 2), 5), ((2, 2, 2), 12), ((3, 3, 3), 8), ((8, 8, 8), 5)])
def test_reported_size_runs(monkeypatch, sub, e):
    print("case: reported size", sub, e, flush=True)
    spec = spec_of(sub, (e, e, e))
    tuned, size = apply_F(spec)
    monkeypatch.setenv("ESPRESO_AUTOTUNE", "0")
    plain, default = apply_F(spec)
    assert default == 320 * 1024

    def fixed(item):
        monkeypatch.setenv("ESPRESO_SYMV_ITEM", str(item))
        y, reported = apply_F(spec)
        assert reported == item
        return y

    assert np.array_equal(plain, fixed(default))
    assert any(np.array_equal(tuned, fixed(item)) for item in (FINE if size == FINE[0] else (size,)))


def test_larger_operator_is_tuned(monkeypatch, capfd):
    """27 and then 64 subdomains of one box (the largest interface 1680 DOFs in both): each is timed once."""
    print("case: larger operator", flush=True)
    monkeypatch.setenv("ESPRESO_MEASURE", "1")
    timed = []
    for n in (3, 3, 4, 4):
        capfd.readouterr()
        apply_F(spec_of((n, n, n), (9, 9, 11)))
        timed.append(capfd.readouterr().err.count("SYMV items tuned"))
    assert timed == [1, 0, 1, 0]
