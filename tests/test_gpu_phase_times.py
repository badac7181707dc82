"""GPU: time_pcg ends where the PCG's work on the device ends.  Without a preconditioner and with
one iteration the PCG applies F twice, to the initial lambda and to the search direction; the second
apply starts after the iteration's stop test is known to the host, so a clock read then would leave
it to the primal recovery's time."""
import warnings

import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


def test_pcg_time_holds_the_last_apply():
    print("case: time of the last apply", flush=True)
    # F of 512 subdomains of 8^3 elasticity: 2.4 GB, 0.37 ms an apply; what else an iteration does takes 0.2 ms
    spec = PB.scaled(PB.GRAVITY, clusters=(8, 8, 8), domains=(1, 1, 1), elements=(8, 8, 8))
    with core.GridFETI(spec, preconditioner="none", max_iterations=1) as g, warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        g.setup()
        apply_s = min(g.time_apply(0, 20)[0] for _ in range(3)) * 1e-3
        pcg_s = min(g.solve()["time_pcg"] for _ in range(5))
        print("apply", apply_s, "pcg", pcg_s, flush=True)
        assert pcg_s >= 2 * apply_s
