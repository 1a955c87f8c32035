"""The autotuner and runs with LDS-resident blocks, which exist at block 256
alone (host side, no kernel launches)."""
import pytest

import parallellbmcranfield_amd as lbm
from parallellbmcranfield_amd import sweep as SW


@pytest.mark.parametrize("prec,instances", [(lbm.PREC_F32, None), (lbm.PREC_F16, None),
                                            (lbm.PREC_F32, [object()])])
@pytest.mark.parametrize("rows", [(0,), (0, 4)])
@pytest.mark.parametrize("winner", [256, 512])
def test_the_default_launches_compete_whatever_block_wins_single_steps(monkeypatch, prec, instances,
                                                                       rows, winner):
    def timer(case, o, inst, steps):
        assert inst is instances
        multi = not o.tune_flags & lbm.TUNE_NO_TWO_STEP
        lds = 5 if multi and o.block_size == 256 and not o.two_step_rows and not o.three_step_rows else 0
        t = (1.0 if o.block_size == winner else 1.01) + 0.001 * o.xcd_group
        tiles = dict(cells=0, tiles=0, rows=0, band=0)
        two = dict(tiles, cells=9 if multi and o.two_step_rows else 0, rows=o.two_step_rows)
        return t * (0.4 if lds else 0.8 if two["cells"] else 1.0), dict(two, lds_steps=lds), tiles

    monkeypatch.setattr(SW, "_time_steps", timer)
    o = lbm.make_options(precision=prec, uavg=0.05, viscosity=0.03)
    best, tried = SW.autotune(None, o, instances=instances, steps=12, blocks=(256, 512),
                              groups=(1, 4), two_rows=rows)
    assert (best["block_size"], best["xcd_group"], best["steps_per_launch"]) == (256, 1, 5)
    assert best["two_step_rows"] == 0 and not best["tune_flags"] & lbm.TUNE_NO_TWO_STEP
    assert sum(r["steps_per_launch"] == 5 for r in tried) == 1


@pytest.mark.parametrize("blocks,rows", [((512,), (0,)), ((256, 512), (4,))])
def test_blocks_and_rows_are_taken_as_asked(monkeypatch, blocks, rows):
    """Without block 256, or without the library's own pick among the rows."""
    calls = []

    def timer(case, o, inst, steps):
        calls.append((o.block_size, o.two_step_rows))
        tiles = dict(cells=0, tiles=0, rows=0, band=0)
        return 1.0 if o.block_size == 512 else 1.01, dict(tiles, lds_steps=0), tiles

    monkeypatch.setattr(SW, "_time_steps", timer)
    best, _ = SW.autotune(None, lbm.make_options(uavg=0.05, viscosity=0.03), steps=12,
                          blocks=blocks, groups=(4,), two_rows=rows)
    assert best["block_size"] == 512
    assert calls == [(b, 0) for b in blocks] + [(512, r) for r in rows] + [(512, 0)]
