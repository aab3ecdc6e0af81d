"""FBP filtering of rows that a fraction of a tile holds, against float64 in
torch: products and sums are float64, the result rounds once, 2^-24: bar 1.2e-7
relative L2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 15, 16, 17, 67])
@pytest.mark.parametrize("nu", [1, 7, 16, 31, 32, 33, 63, 64, 65, 127, 128, 129])
def test_filter(rows, nu):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    r = np.random.default_rng(nu * 100 + rows)
    x, t, w = (torch.from_numpy(r.normal(size=s).astype(np.float32)).cuda() for s in ((rows, nu), nu, nu))
    weighted = rows % 2 == 0
    out = torch.full((rows + 1, nu), 7.0, device="cuda")
    _lib.check(_lib.lib().vir_fbp_filter(_lib.ptr(x), rows, nu, _lib.ptr(w) if weighted else None, _lib.ptr(t),
                                         _lib.ptr(out), stream()), "vir_fbp_filter")
    i = torch.arange(nu, device="cuda")
    ref = (x * w if weighted else x).double() @ t.double()[(i[:, None] - i[None, :]).abs()]
    assert float((out[:rows].double() - ref).norm() / ref.norm()) <= 1.2e-7
    assert bool((out[rows] == 7.0).all())
