"""The host table builder on several worker threads (it takes one per 16384
sites): the same tables as the oracle's whatever the block size and the order
of the records, and the same refusals, naming the lowest site."""
import numpy as np
import pytest

import hemepure_amd as H
import oracle as O
from fixtures import closed_box, sparse_blob


def _lattice(g):
    io = lambda n: [H.iolet_desc(H.COSINE, (0, 0, 0), (0, 0, n))]  # noqa: E731
    return H.Lattice(g, H.params(), io(1), io(-1))


def _shuffled(g, seed):
    o = np.random.default_rng(seed).permutation(g.n_sites)
    return H.Geometry(g.blocks, g.coords[o], g.link_type[o], g.link_iolet[o], g.link_dist[o], g.normal_avail[o],
                      g.normal[o], g.iolets, g.block_size)


@pytest.mark.parametrize("geom", [closed_box(40, 40, 33), sparse_blob(48, spheres=9, block_size=6),
                                  sparse_blob(50, spheres=9, block_size=1)], ids=["box", "blob6", "blob1"])
def test_tables_of_shuffled_records_match_oracle(geom):
    assert geom.n_sites > 2 * 16384
    g = _shuffled(geom, 3)
    lat, ol = _lattice(g), O.OracleLattice(g)
    np.testing.assert_array_equal(lat.class_counts(), ol.class_counts())
    np.testing.assert_array_equal(lat.site_coords(), ol.site_coords())
    push, pull = lat.neighbour_tables()
    np.testing.assert_array_equal(push, ol.push_table())
    for a, b in zip(lat.site_masks(), ol.site_masks()):
        np.testing.assert_array_equal(a, b)
    for a, b in zip(lat.wall_geometry(), (ol.wall_distances(), ol.wall_normals())):
        np.testing.assert_array_equal(a, b)
    # the pull table inverts the push table on plain links
    n, k = lat.n, np.arange(lat.n)
    for j in range(1, 19):
        plain = pull[j - 1] != k
        assert (push[pull[j - 1][plain], j] == k[plain] * 19 + j).all()
    assert n == geom.n_sites


def test_refusals_name_the_lowest_site():
    g = closed_box(40, 40, 33)
    order = _lattice(g).site_coords()
    at = {tuple(c): i for i, c in enumerate(g.coords)}
    late, early = at[tuple(order[30000])], at[tuple(order[20000])]
    for first in (late, early):
        g.link_type[first, 4] = H.LINK_WALL
        with pytest.raises(H.HlbError, match="link type disagrees with neighbour fluidity") as e:
            _lattice(g)
    # two inconsistent links: their sites are wall sites now, behind all bulk
    # sites, so the lowest site is a bulk neighbour on a link's other side
    named = tuple(int(v) for v in str(e.value).split("(")[1].split(")")[0].split(","))
    rank = {tuple(c): i for i, c in enumerate(order)}
    assert named == min((tuple(g.coords[s] + (0, 0, 1)) for s in (late, early)), key=lambda c: rank[c])

    def broken(edit):
        b = closed_box(40, 40, 33)
        edit(b)
        return b

    def duplicate(b):
        b.coords[44000] = b.coords[17]

    def outside(b):
        b.coords[44000] = (0, -1, 0)

    def unknown(b):
        b.link_type[44000, 3] = 9

    for edit, text in ((duplicate, "duplicate fluid site"), (outside, "site outside the block grid"),
                       (unknown, "unknown link type")):
        with pytest.raises(H.HlbError, match=text):
            _lattice(broken(edit))
