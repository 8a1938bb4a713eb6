"""Vessels enumerated in sections along their longest axis (automatic order,
distributions of 64 to 256 MB, longest along y or z): the device's addressing
against the host pull table, and the steps against the same lattice in tile
order, bit for bit."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import Case, W, closed_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,precision", [((13, 60, 301), H.FP64), ((11, 333, 63), H.FP64),
                                           ((30, 41, 400), H.FP32_SHIFTED), ((301, 60, 13), H.FP64)])
def test_sections_address_and_step_like_tiles(box, precision):
    case = Case(closed_box(*box), kernel=H.KERNEL_TRT, wall_bc=H.WALL_BFL, tau=0.7)
    n = case.geom.n_sites
    bytes_ = n * 38 * (8 if precision == H.FP64 else 4)
    assert 64 << 20 < bytes_ <= 256 << 20
    auto = case.product(precision=precision)
    host = auto.neighbour_tables()[1]
    f0 = W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))
    auto.upload_f(f0)
    assert np.array_equal(auto.neighbour_tables()[1], host)
    tile = case.product(precision=precision, slab_order=H.ORDER_TILE)
    tile.upload_f(f0)
    for lat in (auto, tile):
        lat.step(5, properties=True)
    assert np.array_equal(auto.download_f(), tile.download_f())
    for a, b in zip(auto.fields(), tile.fields()):
        assert np.array_equal(a, b)
