"""hlb_device_bytes, by which the server admits requests, covers what a lattice
holds: per site the three distribution sets, fields and site -> slot index, per slab
its record, per boundary and iolet site its arrays, the rows of a sequence of steps
and both buffers of Windkessel terms."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import closed_box, windkessel_cylinder_case


def _bytes(lat):
    return H.lib().hlb_device_bytes(lat._h)


@pytest.mark.parametrize("precision,size", [(H.FP64, 8), (H.FP32_SHIFTED, 4)])
def test_aligned_box(precision, size):
    g = closed_box(64, 64, 64)
    g.coords[:] += 7  # 8..71: every slab is full, so there are as many slots as sites
    lat = H.Lattice(g, H.params(precision=precision), [], [])
    n = lat.n
    wall, iolet, _, _ = lat.site_masks()
    assert n == 64 ** 3 and not iolet.any()
    held = 3 * 19 * size * n + 5 * 8 * n + 4 * n + 256 * (n // 64)
    held += (16 + 18 * 4 + 3 * 4) * int((wall != 0).sum())
    held += 8 * (64 + 1024 * 4)  # the staging's head, 1024 rows of one iolet's three values and the sponge's time
    assert held <= _bytes(lat) <= 1.01 * held


def test_windkessel_terms_are_counted_twice():
    case = windkessel_cylinder_case(kind=H.WK3, radius=10.5, length=17, box_xy=24)
    lat = case.product()
    _, iolet, ids, types = lat.site_masks()
    normal = np.asarray(case.outlets[0].normal)
    d = 5 if normal[2] < 0 else 6  # the link against the outlet's inward normal
    coupled = int(((types == 3) & ((iolet >> (d - 1)) & 1 == 1)).sum())
    assert coupled > 200
    case.outlets[0].kind = H.COSINE
    case.outlets[0].density_mean = 1.0
    plain = case.product()
    assert _bytes(lat) - _bytes(plain) == 16 * (coupled - 1)
