"""Which path a CIC paint takes, by its workspace (host only)."""
import ctypes

import pytest

from bskit_amd import _lib as L


def workspace(N, npart):
    n = L.size_out()
    L.call('bsk_cic_workspace', N, npart, ctypes.byref(n))
    return n.value


@pytest.mark.skipif(not L.built(), reason='libbskhip.so not built')
def test_one_tile_of_many_particles():
    """A tile that is its own neighbour reads up to eight records per particle:
    32-bit counts of them hold below 2^29 particles."""
    assert workspace(16, (1 << 29) - 1) > (1 << 29) * 16  # a record each
    assert workspace(16, 1 << 29) == 16 ** 3 * 8          # atomics
    assert workspace(32, 1 << 29) > (1 << 29) * 16
    assert workspace(40, 1 << 20) == 40 ** 3 * 8
