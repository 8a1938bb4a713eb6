"""An autotuning call that fails leaves the lattice's launch variant as it was:
reported, and chosen anew with the lattice's size unless one had been set."""
import pytest

import hemepure_amd as H
from fixtures import closed_box


def test_failed_autotune_keeps_the_variant():
    large = closed_box(100, 100, 100)  # FP64 planes beyond the Infinity Cache, FP32 ones within
    lat = H.Lattice(large, H.params(), [], [])
    default = lat.variant()
    with pytest.raises(H.HlbError, match="no initial condition"):
        lat.autotune(2)
    assert lat.variant() == default
    p = lat.get_params()
    p.precision = H.FP32_SHIFTED
    lat.set_params(p)
    assert lat.variant() == 1
    lat.set_variant(7)
    with pytest.raises(H.HlbError, match="no initial condition"):
        lat.autotune(2)
    assert lat.variant() == 7
