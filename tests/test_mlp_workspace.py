"""Room the training step takes (CPU: the library's size function alone).  A point needs its three
layers' pre-activations in fp32 and their activations in BF16 in both orders, 6,144 bytes, and
under 60 bytes of outputs and partial sums; gradients take no arrays of their own.  The split-K
partials of two weight gradients are a constant beyond 32,768 points."""
import ctypes
import os

import pytest


@pytest.fixture(scope="module")
def size():
    from streamsculptor_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        from streamsculptor_amd.build import build
        build(verbose=False)
    f = ctypes.CDLL(_lib.LIB_PATH).ssc_mlp_workspace_bytes
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int64]
    return f


@pytest.mark.parametrize("a,b", [(1 << 16, 1 << 20), (100_001, 1 << 24)])
def test_bytes_a_point(size, a, b):
    assert 6144 * (b - a) <= size(b) - size(a) <= 6204 * (b - a)


def test_constant_part(size):
    for n in (1, 63, 300, 512, 8192, 1 << 16):
        assert size(n) <= 6204 * n + 2 * 64 * 256 * 256 * 4
