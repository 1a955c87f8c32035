"""Runs of plain steps with LDS-resident blocks (the default where a lattice
has no open outlets) against every step its own launch (LBM_TUNE_NO_TWO_STEP):
the same fields and distributions bit for bit.  Lattices below, at and above
the block's output rows and columns, for each region shape the library picks
by size, with every class of node (interior, in-tile walls, lid, curved walls,
west inlet, pressure and velocity outlets) and runs of every length up to two
launches."""
import numpy as np
import pytest

import parallellbmcranfield_amd as lbm

pytestmark = pytest.mark.gpu

STORES = [(p, c) for p in (lbm.PREC_F64, lbm.PREC_F32, lbm.PREC_F16, lbm.PREC_F16_SR)
          for c in (lbm.BGKW, lbm.TRT, lbm.MRT)]


def compare(case, chunks, **kw):
    out = []
    for flags in (0, lbm.TUNE_NO_TWO_STEP | lbm.TUNE_NO_THREE_STEP):
        s = lbm.Solver(case, lbm.make_options(rho_ini=1.0, init=lbm.INIT_REST, use_stop_rule=0,
                                              tune_flags=flags, **kw))
        assert (s.lds_steps > 0) == (flags == 0)
        for k in chunks:
            assert s.step(k) == k
        out.append((s.macro(), s.distributions(), s.force_history(), s.residual_history()))
        s.close()
    a, b = out
    for x, y in zip(a[0] + a[1] + a[2] + a[3], b[0] + b[1] + b[2] + b[3]):
        assert np.array_equal(x, y)
    assert np.isfinite(a[0][1]).all() and np.abs(a[0][1]).max() > 0


@pytest.mark.parametrize("prec,coll", STORES)
@pytest.mark.parametrize("nx,ny", [(2, 2), (4, 19), (20, 4), (21, 5), (61, 47), (190, 140)])
def test_small_cavities(prec, coll, nx, ny):
    print("lds small", prec, coll, nx, ny, flush=True)
    compare(lbm.Case.cavity_ex(nx, ny), (1, 2, 3, 4, 9, 15, 7), collision=coll, precision=prec,
            uavg=0.1, viscosity=0.04, resid_kind=lbm.RESID_VELOCITY, resid_every=13)


@pytest.mark.parametrize("prec,coll,nx,ny", [
    (*sc, *n) for sc in STORES for n in ((1000, 480), (1120, 1105))
    if (*sc, *n) != (lbm.PREC_F32, lbm.BGKW, 1120, 1105)])
def test_large_cavities(prec, coll, nx, ny):
    """The regions of larger lattices: an obstacle, uneven sides."""
    print("lds large", prec, coll, nx, ny, flush=True)
    case = lbm.Case.cavity_ex(nx, ny, [(300, 200, 355, 231)])
    compare(case, (23, 2, 3, 12), collision=coll, precision=prec, uavg=0.1, viscosity=0.04,
            trt_lambda=0.25, trt_fp64_parts=1, resid_kind=lbm.RESID_NONE)


@pytest.mark.parametrize("prec,coll", STORES)
@pytest.mark.parametrize("nx,ny,d,extra", [
    (130, 41, 9.0, dict(curved=1, inlet_profile=1, outlet_profile=4)),
    (131, 40, 9.0, dict(curved=2, inlet_profile=1, outlet_profile=4)),
    (90, 33, 0.0, dict(curved=2, inlet_profile=2, outlet_profile=1)),
    (1210, 400, 60.0, dict(curved=1, inlet_profile=1, outlet_profile=4))])
def test_channels(prec, coll, nx, ny, d, extra):
    """Curved and straight cylinder walls, parabolic and uniform inlets,
    pressure and velocity outlets, a force sampled between runs."""
    print("lds channel", prec, coll, nx, ny, extra, flush=True)
    case = lbm.Case.channel(nx, ny, nx / 3 + 0.2, ny / 2 + 0.3, d / 2)
    compare(case, (41, 6), collision=coll, precision=prec, uavg=0.03, viscosity=0.03,
            force_id=5 if d else 0, force_every=11, resid_kind=lbm.RESID_FULL, resid_every=17,
            **extra)


@pytest.mark.parametrize("coll", [lbm.BGKW, lbm.TRT, lbm.MRT])
@pytest.mark.parametrize("nx,ny", [(621, 660), (905, 898)])
def test_wide_fp64_blocks(coll, nx, ny):
    """Blocks of 64 x 32 nodes in registers beside 32 x 32 ones: an obstacle
    inside, sides that leave a part of a wide block."""
    print("lds wide", coll, nx, ny, flush=True)
    compare(lbm.Case.cavity_ex(nx, ny, [(300, 200, 355, 231)]), (21, 3, 2, 9), collision=coll,
            precision=lbm.PREC_F64, uavg=0.1, viscosity=0.04, trt_lambda=0.25, trt_fp64_parts=1,
            resid_kind=lbm.RESID_NONE)


@pytest.mark.parametrize("prec", [lbm.PREC_F32, lbm.PREC_F16, lbm.PREC_F16_SR])
@pytest.mark.parametrize("coll", [lbm.BGKW, lbm.TRT, lbm.MRT])
@pytest.mark.parametrize("nx,ny", [(640, 631), (905, 898), (1290, 1270), (1745, 1731)])
def test_low_precision_blocks_in_registers(prec, coll, nx, ny):
    """The sizes around which the block shapes change; a residual cuts the runs."""
    if coll == lbm.BGKW and prec == lbm.PREC_F32 and nx > 1000:
        pytest.skip("takes two-step launches")
    print("lds registers", prec, coll, nx, ny, flush=True)
    compare(lbm.Case.cavity_ex(nx, ny, [(300, 200, 355, 231)]), (23, 3), collision=coll,
            precision=prec, uavg=0.1, viscosity=0.04, trt_lambda=0.25, trt_fp64_parts=1,
            resid_kind=lbm.RESID_VELOCITY, resid_every=10)


def test_fp32_bgk_with_two_step_launches_keeps_them():
    """Its two-step kernel rounds differently from the single step: the fields
    stay those of these launches."""
    out = []
    for flags in (0, lbm.TUNE_NO_THREE_STEP):
        s = lbm.Solver(lbm.Case.cavity_ex(1120, 1105), lbm.make_options(
            rho_ini=1.0, init=lbm.INIT_REST, use_stop_rule=0, collision=lbm.BGKW,
            precision=lbm.PREC_F32, uavg=0.1, viscosity=0.04, resid_kind=lbm.RESID_NONE,
            tune_flags=flags))
        assert s.lds_steps == 0
        s.step(21)
        out.append(s.distributions())
        s.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("coll", [lbm.BGKW, lbm.TRT, lbm.MRT])
def test_a_force_step_rounds_as_the_residual_kernels_do(coll):
    """Sampling the force alone, or with a residual at the same steps: the
    same fields and forces bit for bit."""
    out = []
    for resid in (lbm.RESID_NONE, lbm.RESID_FULL):
        s = lbm.Solver(lbm.Case.channel(149, 44, 50.2, 22.3, 5.0), lbm.make_options(
            rho_ini=1.0, init=lbm.INIT_REST, use_stop_rule=0, collision=coll,
            precision=lbm.PREC_F32, uavg=0.03, viscosity=0.03, force_id=5, force_every=10,
            resid_kind=resid, resid_every=10, curved=1, inlet_profile=1, outlet_profile=4))
        s.step(61)
        out.append((*s.macro(), s.force_history()[1]))
        s.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))


def test_scale_that_is_no_power_of_two_and_open_outlets_keep_single_steps():
    case = lbm.Case.cavity(40)
    s = lbm.Solver(case, lbm.make_options(precision=lbm.PREC_F16, f16_scale=3000.0))
    assert s.lds_steps == 0
    s.close()
    s = lbm.Solver(lbm.Case.channel(60, 20), lbm.make_options(outlet_profile=2, inlet_profile=1))
    assert s.lds_steps == 0
    s.close()


def test_packed_instance_with_fluid_in_its_outermost_cells_keeps_single_steps():
    i, j = (a.ravel() for a in np.meshgrid(np.arange(6), np.arange(5)))
    nodes = np.stack([i, j, i * 0.1, j * 0.1, np.ones_like(i)], 1)
    edge = lbm.Case.from_arrays(nodes, np.zeros((0, 7)))
    for cases, on in (((lbm.Case.cavity(9), edge), False), ((lbm.Case.cavity(9),) * 2, True)):
        s = lbm.Solver(lbm.Case.pack(cases), lbm.make_options(precision=lbm.PREC_F32),
                       instances=[(0.05, 0.1)] * 2)
        assert (s.lds_steps > 0) == on
        s.close()
