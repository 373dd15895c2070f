"""Orbits that start all along the grid among many sources: the last sizes with a wave per orbit
and the first with lane groups, for each range of the table's size; against the oracle, as the other
launch shapes."""
import pytest

import test_gpu_leapfrog_lanes as lanes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,m,n", [
    ("static", 127, 1025), ("line", 128, 2048), ("line", 128, 2049), ("static", 256, 2560),
    ("tracked", 300, 2561), ("static", 512, 2500), ("static", 513, 2048), ("static", 513, 2049),
])
def test_ragged_shapes(oracle, ssc, kind, m, n):
    lanes.test_launch_shapes(oracle, ssc, kind, m, n, 24)
