"""Joseph backprojection of a grid with more samples a ray than float32 counts
exactly: such grids go to the per-voxel kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_samples_than_float32_counts():
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    from vir_amd.sys_mat.rd import RDProjector
    d = 2e4                                      # a diagonal of 8.02 million units, samples every half unit
    P = RDProjector((2, 401), np.array([0.7, np.pi / 2]), 21, "par", du=2e4, d_pix=d, joseph=True)
    y = torch.full(P.sino_shape, 2.0, device="cuda")
    a, b = P.bp(y), torch.empty(P.img_shape, device="cuda")
    _lib.check(_lib.lib().vir_rd_bp(P.g, _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(y), _lib.ptr(b), 1.0,
                                    _lib.VIR_PER_OUTPUT, stream()), "vir_rd_bp")
    assert torch.equal(a, b) and float(a.max()) > 0
