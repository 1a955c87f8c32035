"""The steps that a launch of LDS-resident blocks makes follow the runs of plain
steps that sampled forces leave: force_every where a force step is a plain one,
one less where it is a residual step (FP32 BGK and TRT)."""
import pytest

import parallellbmcranfield_amd as lbm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coll,every,steps", [
    (lbm.MRT, 5, 5), (lbm.TRT, 5, 4), (lbm.BGKW, 5, 4),  # runs of 5; of 4
    (lbm.MRT, 6, 4), (lbm.TRT, 6, 5),                    # runs of 6; of 5
    (lbm.MRT, 8, 4), (lbm.TRT, 9, 4)])                   # runs of 8
def test_steps_per_launch(coll, every, steps):
    print("force runs", coll, every, steps, flush=True)
    s = lbm.Solver(lbm.Case.channel(1210, 400, 400.2, 200.3, 30.0), lbm.make_options(
        precision=lbm.PREC_F32, collision=coll, rho_ini=1.0, uavg=0.03, viscosity=0.03,
        force_id=5, force_every=every, resid_kind=lbm.RESID_NONE, use_stop_rule=0, curved=1,
        inlet_profile=1, outlet_profile=4))
    assert s.lds_steps == steps
    s.close()
