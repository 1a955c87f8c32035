"""The force that k_force forms ahead of a plain step against the residual form
of the step, which split launches keep: the same fields bit for bit, and forces
that differ by the order of their sums alone.  Bodies in one run of 256
boundary-list nodes, in several rounds of four runs with a part of the last, in
the most runs that take k_force (sixteen) and in more."""
import numpy as np
import pytest

import parallellbmcranfield_amd as lbm

pytestmark = pytest.mark.gpu

# storages and collisions whose force steps are plain steps
FORMS = [(lbm.PREC_F64, lbm.BGKW), (lbm.PREC_F64, lbm.TRT), (lbm.PREC_F64, lbm.MRT),
         (lbm.PREC_F32, lbm.MRT), (lbm.PREC_F16, lbm.MRT), (lbm.PREC_F16_SR, lbm.MRT)]


@pytest.mark.parametrize("prec,coll", FORMS)
@pytest.mark.parametrize("curved", [1, 2])
@pytest.mark.parametrize("nx,ny,r,body", [
    (149, 44, 5.0, 5),     # a cylinder
    (700, 500, 190.0, 5),  # one whose nodes lie among the walls' in many runs
    (1400, 12, 0.0, 4),    # the lower wall: six runs
    (4090, 9, 0.0, 4),     # sixteen
    (4200, 9, 0.0, 4)])    # seventeen: the residual form
def test_force_pass_equals_the_residual_form(prec, coll, curved, nx, ny, r, body):
    print("force forms", prec, coll, curved, nx, ny, body, flush=True)
    case = lbm.Case.channel(nx, ny, nx / 3 + 0.2, ny / 2 + 0.3, r)
    nodes = int((case.cells()["boundary_id"] == body).sum())
    rng = np.random.default_rng(7)  # a flow that reaches every link from the first step on
    rho = 1.0 + 0.02 * rng.standard_normal((case.m, case.n))
    u, v = 0.02 * rng.standard_normal((2, case.m, case.n)) + 0.01
    out = []
    for flags in (0, lbm.TUNE_SPLIT_BOUNDARY):
        s = lbm.Solver(case, lbm.make_options(
            rho_ini=1.0, init=lbm.INIT_FIELD, use_stop_rule=0, collision=coll, precision=prec,
            uavg=0.03, viscosity=0.03, force_id=body, force_every=7, resid_kind=lbm.RESID_NONE,
            curved=curved, inlet_profile=1, outlet_profile=4, tune_flags=flags),
            field=(rho, u, v))
        assert (s.lds_steps > 0) == (flags == 0)
        assert s.step(40) == 40 and s.step(5) == 5
        out.append((s.macro(), s.force_history()))
        s.close()
    (fa, (ia, a)), (fb, (ib, b)) = out
    assert all(np.array_equal(x, y) for x, y in zip(fa, fb))
    assert np.array_equal(ia, ib) and len(ia) == 6
    # at most eight links a node of at most 0.25 each; 8 additions in a lane, 6 in its
    # wave, 4 in its run, 4 over runs and 8 in the tree, twice
    assert np.abs(a - b).max() <= 2 * 30 * 2.0 ** -53 * 8 * 0.25 * nodes
    assert np.isfinite(a).all() and (np.abs(a).max(axis=0) > 1e-4).all()


@pytest.mark.parametrize("prec,coll", FORMS)
@pytest.mark.parametrize("every,resid,resid_every", [
    (1, lbm.RESID_NONE, 1), (2, lbm.RESID_FULL, 2), (4, lbm.RESID_VELOCITY, 2),
    (6, lbm.RESID_FULL, 4), (2, lbm.RESID_REFERENCE, 1)])
def test_force_of_an_evaluated_step(prec, coll, every, resid, resid_every):
    """Forces of every step, and of steps that are evaluated too, some or all of
    them: rows in order, equal to the split launches'."""
    print("force of evaluated steps", prec, coll, every, resid, resid_every, flush=True)
    case = lbm.Case.channel(60, 149, 20.2, 75.3, 9.0)  # the reference residual's cells hold nodes
    nodes = int((case.cells()["boundary_id"] == 5).sum())
    rng = np.random.default_rng(7)
    rho = 1.0 + 0.02 * rng.standard_normal((case.m, case.n))
    u, v = 0.02 * rng.standard_normal((2, case.m, case.n)) + 0.01
    out = []
    for flags in (0, lbm.TUNE_SPLIT_BOUNDARY):
        s = lbm.Solver(case, lbm.make_options(
            rho_ini=1.0, init=lbm.INIT_FIELD, use_stop_rule=0, collision=coll, precision=prec,
            uavg=0.03, viscosity=0.03, force_id=5, force_every=every, resid_kind=resid,
            resid_every=resid_every, curved=1, inlet_profile=1, outlet_profile=4,
            tune_flags=flags), field=(rho, u, v))
        assert s.step(40) == 40
        out.append((s.macro(), s.force_history(), s.residual_history()))
        s.close()
    (fa, (ia, a), (ra, va)), (fb, (ib, b), (rb, vb)) = out
    assert all(np.array_equal(x, y) for x, y in zip(fa, fb))
    assert np.array_equal(ia, ib) and np.array_equal(ia, np.arange(every - 1, 40, every))
    assert np.array_equal(ra, rb)
    assert len(ra) == (0 if resid == lbm.RESID_NONE else 40 // resid_every)
    assert np.abs(a - b).max() <= 2 * 30 * 2.0 ** -53 * 8 * 0.25 * nodes
    if len(ra):
        assert np.allclose(va, vb, rtol=1e-12, atol=0)
