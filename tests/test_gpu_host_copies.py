"""GPU: host vectors that cross through pinned chunks: exactly the smallest such size
(64^3 doubles, 2 MB), one with a ragged last chunk (65^3) and one with more
chunks than slots (131^3, 18 MB), from pageable and from pinned memory, and two
threads with an instance each.

Bar: nodal loads come back to 2 units in the last place (they are split over up
to 8 copies of a node and summed again).
"""
import sys
import threading

import numpy as np
import pytest
import torch

from espreso_amd import core

pytestmark = pytest.mark.gpu


def heat(subs, e):
    return dict(physics=1, clusters=(subs, subs, subs), domains=(1, 1, 1), elements=(e, e, e), length=(1.0, 1.0, 1.0),
                conductivity=2.0, heat_source=1.0, fixed=(0, 0, 0, 0, 1, 0))


def roundtrip(g, load):
    g.set_nodal_rhs(load)
    assert np.all(np.abs(g.nodal_load() - load) <= 2 * np.spacing(np.abs(load)))


@pytest.mark.parametrize("subs,e", [(7, 9), (8, 8), (13, 10)])
def test_sizes(subs, e):
    print("case: host copies", subs, e, flush=True)
    sys.stdout.flush()
    g = core.GridFETI(heat(subs, e))
    g.setup()
    n = (subs * e + 1)**3
    rng = np.random.default_rng(31)
    for _ in range(2):
        roundtrip(g, rng.standard_normal((n, 1)))
    pinned = torch.empty((n, 1), dtype=torch.float64, pin_memory=True).numpy()
    pinned[:] = rng.standard_normal((n, 1))
    roundtrip(g, pinned)
    g.close()


def test_threads():
    bad = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            for _ in range(2):  # the second instance has streams of its own
                g = core.GridFETI(heat(8, 8))
                g.setup()
                for _ in range(4):
                    roundtrip(g, rng.standard_normal((65**3, 1)))
                g.close()
        except BaseException as e:  # noqa: BLE001
            bad.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
