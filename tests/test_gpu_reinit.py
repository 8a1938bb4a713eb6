"""A lattice whose first device state could not be made is configured anew, with
more iolets, and then runs as a lattice made that way from the start: what it
stages per step is sized for the iolets it has then."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import four_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [H.FP64, H.FP32_SHIFTED])
def test_more_iolets_after_a_failed_state(precision):
    g = four_cube(9, seed=2)
    prm = H.params(wall_bc=H.WALL_GZS, tau=0.8, precision=precision)

    def iolets(radius, count):
        inlet = H.iolet_desc(H.PARABOLIC, (4.0, 4.0, 0.5), (0, 0, 1), radius=radius, max_speed=0.01)
        out = H.iolet_desc(H.COSINE, (4.0, 4.0, 7.5), (0, 0, -1), density_mean=0.99, density_amp=2e-3, period=9.0)
        return [inlet], [out] * count

    late = H.Lattice(g, prm, *iolets(1.0, 1))
    with pytest.raises(H.HlbError, match="outside the IOLET radius"):
        late.init_equilibrium(1.0)  # a GZS wall link reads the inlet's profile beyond its radius
    late.set_iolets(*iolets(20.0, 100))
    fresh = H.Lattice(g, prm, *iolets(20.0, 100))
    for lat in (late, fresh):
        lat.init_equilibrium(1.0)
        lat.step(1030, properties=True)  # a full chunk of staged steps and a short one
    assert np.isfinite(fresh.download_f()).all()
    assert np.array_equal(late.download_f(), fresh.download_f())
    assert late.monitor() == fresh.monitor()
