"""FBP: a view without a finite angle adds nothing, whatever the geometry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("geom,DSO", [("par", 0.0), ("flat", 140.0), ("arc", 70.0), ("arc", 350.0), ("arc", 2000.0)])
def test_views_without_an_angle(geom, DSO, bad):
    import torch
    from vir_amd.fbp import FBP
    kw = {} if geom == "par" else dict(DSO=DSO, DSD=1.5 * DSO, du=1.5, detector=geom)
    ang = np.arange(9) * 0.3
    keep = [0, 1, 2, 3, 5, 6, 7]
    some = ang.copy()
    some[[4, 8]] = bad
    y = torch.rand(9, 70, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    P, Q = (FBP((40, 41), a, 70, "par" if geom == "par" else "fan", **kw) for a in (some, ang[keep]))
    a, b = P(y), Q(y[keep].contiguous()) * (7.0 / 9.0)
    # the same float64 sums; float32 rounding of the sum, the scale and 7 / 9
    assert float((a - b).double().norm() / b.double().norm()) <= 2.4e-7
