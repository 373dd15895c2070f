"""Orbits that start all along the grid among many sources: the last sizes with a wave per orbit
and the first with lane groups, for each range of the table's size; and straight-line sources, which
have a rule of their own, with each number of lanes, whole rounds of waves beside a remainder
(starts all at the first row) and pairs of orbits.  Against the oracle, as the other launch shapes."""
import pytest

import test_gpu_leapfrog_lanes as lanes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,m,n", [
    ("static", 127, 1025), ("line", 128, 2048), ("line", 128, 2049), ("static", 256, 2560),
    ("tracked", 300, 2561), ("static", 512, 2500), ("static", 513, 2048), ("static", 513, 2049),
])
def test_ragged_shapes(oracle, ssc, kind, m, n):
    lanes.test_launch_shapes(oracle, ssc, kind, m, n, 24)


@pytest.mark.parametrize("kind,m,n,nsteps", [
    ("line", 30, 1025, 24), ("line", 30, 2048, 24), ("line", 30, 2049, 24),  # wave, wave, 16 lanes
    ("hernquist", 64, 4096, 24), ("hernquist", 64, 4097, 24),
    ("line", 30, 20000, 12), ("hernquist", 31, 40001, 8), ("line", 30, 70000, 6),  # 8, 4, 2 lanes
    ("line", 15, 32767, 8), ("line", 15, 32768, 8),  # few sources: lanes, one lane
    ("line", 30, 200001, 4),                         # the window's shape: three rounds and a remainder
    ("hernquist", 17, 393217, 3),                    # pairs
])
def test_straight_lines(oracle, ssc, kind, m, n, nsteps):
    lanes.test_launch_shapes(oracle, ssc, kind, m, n, nsteps)
