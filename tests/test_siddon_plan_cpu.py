"""View chunks of the Siddon backprojection, seen in its workspace (one partial
volume a chunk, none for one chunk; host rule)."""
import pytest


@pytest.mark.parametrize("n,views,chunks", [
    ((64, 64, 64), 120, 30),      # pairs of views, twice the resident blocks
    ((64, 64, 64), 90, 23),
    ((200, 200, 24), 60, 8),
    ((128, 128, 128), 90, 4),
    ((96, 96, 64), 10, 5),        # two views a chunk, not one
    ((64, 64, 64), 30, 15),
    ((48, 48, 16), 90, 45),
    ((128, 128, 32), 40, 8),      # the chip filled just so
    ((256, 256, 16), 30, 4),
    ((32, 32, 32), 10, 10),       # a single view each, few blocks
    ((256, 256, 256), 360, 1),    # one chunk, no partial volumes
    ((512, 512, 16), 30, 1),
    ((64, 64, 64), 1, 1),
])
def test_chunks(n, views, chunks):
    from vir_amd import _lib
    from vir_amd.sys_mat.siddon import grid_params
    g = _lib.make_grid(*grid_params(n, 1.0, 0.0), 1e-5)
    ws = _lib.lib().vir_siddon_bp_workspace(g, views)
    assert ws == (0 if chunks == 1 else chunks * n[0] * n[1] * n[2] * 4)
