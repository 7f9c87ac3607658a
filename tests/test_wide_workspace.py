"""A workspace sized for some rows (up to 128) serves every call of fewer: the
size that the library asks for never falls as the rows grow, although fewer rows
may be split over more slice groups."""
import ctypes

import pytest

from quipsharp_amd import _lib


@pytest.mark.parametrize("m", [256, 1024, 3584, 4096, 5120, 8192, 11008, 14336, 16384, 18944, 25600, 32768])
@pytest.mark.parametrize("n", [256, 1024, 4096, 14336, 25600])
def test_workspace_grows_with_rows(m, n):
    size = _lib.lib().qs_linear_workspace_bytes
    need = [size(m, n, rows, _lib.QS_LAYOUT_TILED) for rows in range(17, 129)]
    assert need == sorted(need)


def test_workspace_grows_over_every_path():
    """One-launch and 16-row calls, then the wide GEMM through all its splits."""
    size = _lib.lib().qs_linear_workspace_bytes
    for m, n in ((4096, 4096), (11008, 4096), (4096, 14336), (25600, 5120), (1024, 3584), (256, 256), (32768, 512)):
        need = [size(m, n, rows, _lib.QS_LAYOUT_TILED) for rows in range(1, 2050)]
        falls = [rows + 1 for rows in range(1, len(need)) if need[rows] < need[rows - 1]]
        assert not falls, (m, n, falls)


@pytest.mark.parametrize("n,ms", [(4096, (4096, 1024, 1024)), (5120, (25600, 25600)), (3584, (3584, 512, 512))])
def test_group_workspace_grows_with_rows(n, ms):
    sizes = (ctypes.c_int64 * len(ms))(*ms)
    need = [_lib.lib().qs_linear_group_workspace_bytes(n, rows, len(ms), sizes) for rows in range(1, 2050)]
    assert need == sorted(need)
