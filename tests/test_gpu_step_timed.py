"""step_timed's kernel time: the average launch of the kernel that made the
most steps per launch in that call, also where every step is evaluated and the
call makes single-step launches alone."""
import pytest

import parallellbmcranfield_amd as lbm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,prec,coll,steps,every,kw", [
    (64, 64, lbm.PREC_F64, lbm.BGKW, 50, 1, dict(resid_kind=lbm.RESID_VELOCITY, resid_every=1)),
    (64, 64, lbm.PREC_F32, lbm.MRT, 50, 4, dict(resid_kind=lbm.RESID_FULL, resid_every=2)),
    (40, 90, lbm.PREC_F64, lbm.TRT, 30, 1, dict(resid_kind=lbm.RESID_REFERENCE)),
    (64, 64, lbm.PREC_F64, lbm.BGKW, 50, 1, dict(resid_kind=lbm.RESID_NONE)),
    (64, 64, lbm.PREC_F64, lbm.BGKW, 2, 1, dict(resid_kind=lbm.RESID_NONE)),
    (1100, 1100, lbm.PREC_F32, lbm.MRT, 12, 1, dict(resid_kind=lbm.RESID_FULL, resid_every=1)),
    (1100, 1100, lbm.PREC_F32, lbm.MRT, 2, 1, dict(resid_kind=lbm.RESID_NONE)),
    (2100, 2100, lbm.PREC_F32, lbm.MRT, 3, 2, dict(resid_kind=lbm.RESID_NONE))])
def test_kernel_time_of_what_ran(nx, ny, prec, coll, steps, every, kw):
    print("step_timed", nx, ny, prec, coll, steps, every, kw, flush=True)
    s = lbm.Solver(lbm.Case.cavity_ex(nx, ny), lbm.make_options(
        rho_ini=1.0, init=lbm.INIT_REST, use_stop_rule=0, collision=coll, precision=prec,
        uavg=0.05, viscosity=0.04, **kw))
    assert s.lds_steps > 0
    s.step(steps)
    total, kern = s.step_timed(steps, every)
    assert s.iter == 2 * steps
    assert 0 < kern < total
    s.close()
