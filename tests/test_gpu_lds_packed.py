"""LDS-resident blocks on packed lattices of the size whose blocks of interior
nodes are held in registers: uneven cavities with obstacles, their own rates,
some of which stop midway, against every step its own launch."""
import numpy as np
import pytest

import parallellbmcranfield_amd as lbm
from parallellbmcranfield_amd import sweep as SW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lbm.PREC_F32, lbm.PREC_F16, lbm.PREC_F16_SR])
@pytest.mark.parametrize("coll", [lbm.BGKW, lbm.TRT, lbm.MRT])
def test_packed_lattices_equal_single_steps(prec, coll):
    print("lds packed", prec, coll, flush=True)
    # Re below where TRT at these rates diverges from a rest start (about 2000)
    specs = SW.random_cavities(24, seed=5, side=(65, 220), re=(100.0, 800.0))
    packed, _ = SW.build_batch(specs)
    assert 400_000 <= packed.n * packed.m <= 600_000

    def solver(flags, crit):
        return lbm.Solver(packed, lbm.make_options(
            collision=coll, precision=prec, uavg=0.1, rho_ini=1.0, viscosity=0.02,
            init=lbm.INIT_REST, resid_kind=lbm.RESID_VELOCITY, resid_every=23, use_stop_rule=1,
            max_iterations=10**6, crit_v=crit, tune_flags=flags, trt_lambda=0.25,
            trt_fp64_parts=1), instances=[(sp["nu"], sp["lid"]) for sp in specs])

    single = lbm.TUNE_NO_TWO_STEP | lbm.TUNE_NO_THREE_STEP
    s = solver(single, 0.0)
    s.step(230)
    crit = float(np.median(s.batch_status()[2]))  # half of them are below it by then
    s.close()
    out = []
    for flags in (0, single):
        s = solver(flags, crit)
        assert (s.lds_steps > 0) == (flags == 0)
        for k in (100, 1, 57, 142):
            assert s.step(k) == k
        it, _, res = s.batch_status()
        out.append((it, res, s.residual_history()[1], *s.macro(), *s.distributions()))
        s.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))
    stopped = out[0][0] > 0
    assert 4 <= stopped.sum() < len(specs) and len(set(out[0][0][stopped])) > 1
    assert np.isfinite(out[0][4]).all()
