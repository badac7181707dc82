"""GPU: a null host vector is an error of the call at every size (small vectors take the
runtime's copy, those of 2 MB and more the threaded one), and leaves no error behind: the
instance and new ones work on."""
import numpy as np
import pytest

from espreso_amd import core
from espreso_amd import problems as PB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,e,large", [(2, 3, False), (8, 8, True)])
def test_null_vectors(n, e, large):
    print("case: null vectors", n, e, flush=True)
    lib = core.lib()
    with core.GridFETI(PB.scaled(PB.GRAVITY, clusters=(n, n, n), domains=(1, 1, 1), elements=(e, e, e)),
                       preconditioner="lumped") as g:
        g.setup()
        assert (8 * g.n_lambda >= 2 << 20) == large
        x = np.random.default_rng(31).standard_normal(g.n_lambda)
        ref, out = g.apply_F(x), np.empty_like(x)
        for call in (lib.espreso_feti_apply_F, lib.espreso_feti_apply_prec, lib.espreso_feti_project):
            assert call(g.h, None, core._dp(out)) != 0
            assert call(g.h, core._dp(x), None) != 0
        g.solve()
        assert lib.espreso_grid_nodal_solution(g.h, None) != 0
        g.setup()
        assert np.array_equal(g.apply_F(x), ref)
