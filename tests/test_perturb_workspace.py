"""Room the fixed-step responses ask for (CPU: the library's size function alone): two segments of
rows of 72 bytes a particle, an eighth of the grid each and at least 64 rows, all rows of shorter
grids, at most 4 GiB and at least one row."""
import ctypes
import os

import pytest


@pytest.mark.parametrize("n,nsteps,rows", [
    (8000, 4000, 2 * 501),          # 577 MB; all rows would be 2.3 GB
    (1000, 511, 2 * 64), (1000, 512, 2 * 65), (10, 128, 2 * 64),
    (10, 127, 128), (10, 0, 1), (500_000, 100, 101),  # fewer than two segments: all rows
    (80_000, 4000, (1 << 32) // (72 * 80_000)),       # the limit
    (100_000_000, 10, 1),                             # one row, whatever it takes
    (0, 100, 0),
])
def test_rows(n, nsteps, rows):
    from streamsculptor_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        from streamsculptor_amd.build import build
        build(verbose=False)
    f = ctypes.CDLL(_lib.LIB_PATH).ssc_perturb_workspace_bytes
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int64, ctypes.c_int32]
    assert f(n, nsteps) == rows * n * 72
