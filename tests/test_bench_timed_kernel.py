"""bench.py's account of the launches that lbm_solver_step_timed samples, on
the host (no kernel launches)."""
import os
import sys
from types import SimpleNamespace

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench


def solver(lds=0, two=0, three=0):
    return SimpleNamespace(lds_steps=lds, paired=False, fused=True,
                           two_step_info=lambda: dict(cells=two),
                           three_step_info=lambda: dict(cells=three))


def square(n):
    return SimpleNamespace(n=n + 2, m=n + 3, info=SimpleNamespace(num_fluid=n * n, num_boundary=4 * n))


@pytest.mark.parametrize("n,s,steps,every,kernel,made", [
    (4097, solver(5, 9, 9), 20, 1, "k_lds_steps", [5, 5, 5, 4]),
    (4097, solver(5, 9, 9), 4, 1, "k_lds_steps", [3]),
    (4097, solver(5, 9, 9), 3, 1, "k_three_steps", [3]),  # two before the last: no LDS launch
    (4097, solver(5, 9, 9), 2, 1, "k_two_steps", [2]),
    (1100, solver(4, 9, 9), 3, 1, "k_lds_steps", [2]),
    (1100, solver(4, 9, 0), 2, 1, "k_two_steps", [2]),
    (129, solver(7), 2, 1, "k_step", [1, 1]),
    (129, solver(7), 17, 8, "k_lds_steps", [7, 5]),  # steps 0-6, 7-11, 12-15 and the last
    (4097, solver(0, 9, 9), 20, 1, "k_three_steps", [3] * 6),
    (4097, solver(0, 9, 0), 5, 4, "k_two_steps", [2]),
    (129, solver(), 9, 4, "k_step", [1, 1, 1])])
def test_launches_timed(n, s, steps, every, kernel, made):
    _, launches, name = bench.timed_kernel(s, square(n), steps, every)
    assert (name.split()[0], launches) == (kernel, made)
