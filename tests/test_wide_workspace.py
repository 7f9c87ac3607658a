"""A workspace sized for some rows (up to 128) serves every call of fewer: the
size that the library asks for never falls as the rows grow, although fewer rows
may be split over more slice groups."""
import pytest

from quipsharp_amd import _lib


@pytest.mark.parametrize("m", [256, 1024, 3584, 4096, 5120, 8192, 11008, 14336, 16384, 18944, 25600, 32768])
@pytest.mark.parametrize("n", [256, 1024, 4096, 14336, 25600])
def test_workspace_grows_with_rows(m, n):
    size = _lib.lib().qs_linear_workspace_bytes
    need = [size(m, n, rows, _lib.QS_LAYOUT_TILED) for rows in range(17, 129)]
    assert need == sorted(need)
