"""A lattice carries marks for wall and iolet links between two fluid sites exactly if
it has one: a single such link anywhere, in any direction, is found, and geometries
without one, on slabs of every fill, are not taken to have any.  (The marks are one
word per boundary site of the lattice's device bytes.)"""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import CX, CY, CZ, INV, closed_box, sparse_blob


def _bytes(g):
    lat = H.Lattice(g, H.params(), [], [])
    wall, _, _, _ = lat.site_masks()
    return H.lib().hlb_device_bytes(lat._h), (int((wall != 0).sum()) + 63) // 64 * 64


@pytest.mark.parametrize("geom", [closed_box(9, 17, 8), closed_box(1, 9, 13), closed_box(20, 5, 33),
                                  sparse_blob(30, spheres=4, block_size=6), sparse_blob(26, spheres=3, block_size=1)],
                         ids=["box", "sheet", "bar", "blob6", "blob1"])
def test_one_link_is_found_and_none_invented(geom):
    plain, words = _bytes(geom)
    at = {tuple(c): i for i, c in enumerate(geom.coords.tolist())}
    rng = np.random.default_rng(4)
    wall = (geom.link_type == H.LINK_WALL).any(axis=1)
    for d in range(1, 19):
        # two boundary sites, so that the number of boundary sites stays
        pairs = [(i, at[n]) for i, c in enumerate(geom.coords.tolist())
                 if (n := (c[0] + CX[d], c[1] + CY[d], c[2] + CZ[d])) in at and wall[i] and wall[at[n]]]
        if not pairs:
            continue
        i, k = pairs[rng.integers(len(pairs))]
        geom.link_type[i, d - 1] = geom.link_type[k, INV[d] - 1] = H.LINK_WALL
        assert _bytes(geom) == (plain + 4 * words, words)
        geom.link_type[i, d - 1] = geom.link_type[k, INV[d] - 1] = H.LINK_NONE
    assert _bytes(geom) == (plain, words)
