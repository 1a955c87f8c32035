"""Packed instances one cell wide or high, with and without a node."""
import numpy as np
import pytest

import parallellbmcranfield_amd as lbm

pytestmark = pytest.mark.gpu


def mesh(n, m, fluid):
    i, j = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(m)))
    return lbm.Case.from_arrays(np.stack([i, j, i * 0.1, j * 0.1, fluid], 1), np.zeros((0, 7)))


@pytest.mark.parametrize("n,m,fluid,on", [
    (1, 5, [0, 0, 1, 0, 0], False),  # a node in the outermost cells: single steps
    (1, 5, [0, 0, 0, 0, 0], True),
    (5, 1, [0, 0, 0, 0, 0], True),
    (2, 5, [0] * 10, True),
    (3, 3, [0, 0, 0, 0, 1, 0, 0, 0, 0], True)])
def test_narrow_instances(n, m, fluid, on):
    print("narrow instance", n, m, fluid, flush=True)
    out = []
    for flags in (0, lbm.TUNE_NO_TWO_STEP):
        s = lbm.Solver(lbm.Case.pack([lbm.Case.cavity(9), mesh(n, m, np.array(fluid))]),
                       lbm.make_options(precision=lbm.PREC_F32, rho_ini=1.0, init=lbm.INIT_REST,
                                        use_stop_rule=0, tune_flags=flags),
                       instances=[(0.05, 0.1)] * 2)
        assert (s.lds_steps > 0) == (on and not flags)
        s.step(17)
        out.append((*s.macro(), *s.distributions()))
        s.close()
    # a node between solid cells alone empties, to a density of zero
    assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(*out))
    assert np.nanmax(np.abs(out[0][1])) > 0
