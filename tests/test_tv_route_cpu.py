"""Which images vir_tv_chambolle_pair is chosen for (a host rule)."""
import pytest


@pytest.mark.parametrize("shape,pays", [
    ((256, 256, 256), 1), ((512, 512, 16), 1), ((128, 128, 128), 1), ((1024, 1024), 1), ((128, 128), 1), ((4, 256, 512), 1),
    ((512, 512, 1), 0), ((512, 512, 4), 0), ((512, 1, 512), 0), ((64, 64, 64), 0), ((256, 256, 4), 0), ((200000, 4), 0),
    ((7,), 0), ((0, 4), 0), ((2147483647, 2147483647), 1), ((1, 1, 1), 1),
])
def test_rule(shape, pays):
    from vir_amd import _lib
    assert _lib.lib().vir_tv_pair_pays(len(shape), *(shape + (1,) * (3 - len(shape)))) == pays
