"""Host helpers without a library that loads; libraries of another version."""
import os
import subprocess

import numpy as np
import pytest

from bskit_amd import _lib
from bskit_amd.bins import closed_triangle_indices


@pytest.fixture
def other_library(monkeypatch, tmp_path):
    path = tmp_path / 'libbskhip.so'
    monkeypatch.setattr(_lib, '_lib', None)
    monkeypatch.setattr(_lib, 'LIB_PATH', str(path))
    return path


def compiled(path, source):
    src = path.with_suffix('.c')
    src.write_text(source)
    subprocess.check_call([os.environ.get('CC', 'cc'), '-shared', '-fPIC', str(src), '-o', str(path)])


@pytest.mark.parametrize('kind', ['none', 'not a library', 'needs another', 'other version'])
def test_triangle_list_without_library(other_library, kind):
    if kind == 'not a library':
        other_library.write_bytes(b'text')
    elif kind == 'needs another':  # unresolved symbols: as without a HIP runtime
        compiled(other_library, 'extern int not_there; int *p = &not_there;')
    elif kind == 'other version':
        compiled(other_library, 'int bsk_version(void) { return 1; }')
    k = np.array([[0.25 * i, 0.25 * (i + 1)] for i in range(1, 9)])
    for nf in (1, 2, 3):  # FP32 edges (exact here) go by numpy whatever is built
        assert np.array_equal(closed_triangle_indices(k, nf),
                              closed_triangle_indices(k.astype(np.float32), nf))
    assert not _lib.built()
    with pytest.raises((OSError, ImportError, AttributeError)):
        _lib.lib()  # the kernels have no twin


def test_other_version_is_named(other_library):
    """A library that lacks newer symbols: the version is what is reported."""
    compiled(other_library, 'int bsk_version(void) { return 7; }')
    assert _lib.ABI_VERSION > 7  # 7 was before bsk_closed_triangles and the FP64 pair sums
    with pytest.raises(ImportError, match='ABI version 7'):
        _lib.lib()
