"""Plans that do not fit in host memory: a status, not an abort (host only)."""
import subprocess
import sys

import pytest

from bskit_amd import _lib as L

CODE = """
import ctypes, resource, sys
import numpy as np
from bskit_amd import _lib as L
lib = L.lib()
T, n = 6000000, 60
tri = np.random.default_rng(0).integers(0, n, (T, 3), dtype=np.int32)
level = np.zeros(T, np.int32)
ip = ctypes.POINTER(ctypes.c_int)
t, lv, h = tri.ctypes.data_as(ip), level.ctypes.data_as(ip), ctypes.c_void_p()
calls = {'bsk_blocked_create': (0, n, T, t), 'bsk_pairs_create': (0, n, T, t),
         'bsk_pairs_create_levels': (0, n, T, t, lv), 'bsk_pairs_create_f64': (0, n, T, t, lv),
         'bsk_gridinfo_pairs': (n, T, t)}
used = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (48 << 20), resource.RLIM_INFINITY))
rc = getattr(lib, sys.argv[1])(ctypes.byref(h), *calls[sys.argv[1]])
print(rc, h.value, lib.bsk_last_error().decode())
"""


@pytest.mark.skipif(not L.built(), reason='libbskhip.so not built')
@pytest.mark.parametrize('entry', ['bsk_blocked_create', 'bsk_pairs_create',
                                   'bsk_pairs_create_levels', 'bsk_pairs_create_f64',
                                   'bsk_gridinfo_pairs'])
def test_out_of_memory(entry):
    p = subprocess.run([sys.executable, '-c', CODE, entry], capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0, p.stderr[-500:]
    assert p.stdout.strip() == '%d None %s: out of host memory' % (L.ENOMEM, entry)
