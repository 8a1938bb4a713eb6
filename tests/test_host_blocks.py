"""The host tables whatever the geometry's block size: one-cell blocks, small ones,
blocks so large that they are shared out by layers, and nearly empty ones, which are
checked site by site: the oracle's tables, and the same refusals."""
import numpy as np
import pytest

import hemepure_amd as H
import oracle as O
from fixtures import closed_box, sparse_blob


def _blocks(g, bs, shift=(0, 0, 0)):
    c = g.coords + np.asarray(shift)
    return H.Geometry(tuple(int(v) for v in c.max(0) // bs + 1), c, g.link_type, g.link_iolet, g.link_dist,
                      g.normal_avail, g.normal, g.iolets, bs)


def _lattice(g):
    return H.Lattice(g, H.params(), [], [])


@pytest.mark.parametrize("bs", [1, 2, 3, 7, 16, 17, 32, 64])
@pytest.mark.parametrize("name", ["box", "dot", "blob"])
def test_tables(name, bs):
    g = {"box": lambda: closed_box(9, 5, 12), "dot": lambda: closed_box(1, 1, 2),
         "blob": lambda: sparse_blob(26, spheres=4)}[name]()
    g = _blocks(g, bs, (bs - 2, 0, 3) if bs > 2 else (0, 0, 0))  # across a block's face
    lat, ol = _lattice(g), O.OracleLattice(g)
    np.testing.assert_array_equal(lat.class_counts(), ol.class_counts())
    np.testing.assert_array_equal(lat.site_coords(), ol.site_coords())
    push, pull = lat.neighbour_tables()
    np.testing.assert_array_equal(push, ol.push_table())
    for a, b in zip(lat.site_masks(), ol.site_masks()):
        np.testing.assert_array_equal(a, b)
    k = np.arange(lat.n)
    for j in range(1, 19):
        plain = pull[j - 1] != k
        assert (push[pull[j - 1][plain], j] == k[plain] * 19 + j).all()


@pytest.mark.parametrize("bs", [1, 2, 8, 17, 64])
def test_refusals(bs):
    def broken(edit):
        g = closed_box(9, 5, 12)
        edit(g)
        return _blocks(g, bs)

    def one_sided(g):
        inside = np.flatnonzero((g.coords == (5, 3, 6)).all(axis=1))[0]
        g.link_type[inside, 4] = H.LINK_WALL

    def leak(g):
        g.link_type[np.flatnonzero(g.link_type.any(axis=1))[0]] = H.LINK_NONE

    def duplicate(g):
        g.coords[3] = g.coords[100]

    with pytest.raises(H.HlbError, match=r"disagrees with neighbour fluidity at site \(5,3,7\) direction 6 .*zero"):
        _lattice(broken(one_sided))
    with pytest.raises(H.HlbError, match="disagrees with neighbour fluidity"):
        _lattice(broken(leak))
    with pytest.raises(H.HlbError, match="duplicate fluid site"):
        _lattice(broken(duplicate))
