"""Wall and iolet links between two fluid sites (a wall of no thickness, such as
the septum between two touching branches): the neighbour is there, yet its value
must not cross the link.  Whole septa within a tile and along a tile's face, and
links picked at random in every direction, with walls on both sides, iolets on
both, or one of each; steady, property and general-gather steps and downloads
against the oracle: bitwise in FP64, within the shifted form's tolerance in FP32,
alone and in a batch."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import CX, CY, CZ, INV, Case, W, closed_box, four_cube, sparse_blob, IoletSpec

pytestmark = pytest.mark.gpu

DIST = np.array([0.25, np.nextafter(np.float32(0.5), np.float32(0)), 0.5, 0.9, 1.0], dtype=np.float32)
NONE, WALL, INLET = H.LINK_NONE, H.LINK_WALL, H.LINK_INLET


def _pairs(g):
    """Every plain link once: (site, direction, site it leads to)."""
    at = {tuple(c): i for i, c in enumerate(g.coords.tolist())}
    for i, c in enumerate(g.coords.tolist()):
        for d in range(1, 19, 2):
            k = at.get((c[0] + CX[d], c[1] + CY[d], c[2] + CZ[d]))
            if k is not None and g.link_type[i, d - 1] == NONE:
                yield i, d, k


def _cut(g, pick, rng):
    """Makes the links pick(g, site, direction, other) names into walls or iolets
    from both sides; pick returns the two link types."""
    made = set()
    for i, d, k in list(_pairs(g)):
        types = pick(g, i, d, k)
        if types is None:
            continue
        for s, e, t in ((i, d, types[0]), (k, int(INV[d]), types[1])):
            g.link_type[s, e - 1] = t
            g.link_iolet[s, e - 1] = 0 if t == INLET else -1
            g.link_dist[s, e - 1] = rng.choice(DIST)
            made.add((e, t))
            if t == WALL and not g.normal_avail[s]:
                g.normal_avail[s], g.normal[s] = 1, (0.6, 0.0, 0.8)
    return made


def _plane(x, types):
    return lambda g, i, d, k: types if min(g.coords[i, 0], g.coords[k, 0]) == x != max(g.coords[i, 0], g.coords[k, 0]) \
        else None


def _case(name, wall_bc):
    rng = np.random.default_rng(11)
    kind, bc = IoletSpec(H.COSINE, (6.0, 5.0, 4.0), (1, 0, 0), density_mean=1.01, density_amp=4e-3, period=5.0), H.IOLET_NASH
    outlets = []
    if name == "cube":  # a septum between two branches that share inlet and outlet
        g = four_cube(10, seed=4)
        _cut(g, _plane(4, (WALL, WALL)), rng)
        kind = IoletSpec(H.COSINE, (4.5, 4.5, 0.5), (0, 0, 1), density_mean=1.01)
        outlets = [IoletSpec(H.COSINE, (4.5, 4.5, 8.5), (0, 0, -1), density_mean=0.99)]
    elif name in ("face", "inner", "sheets", "iolets"):
        g = {"sheets": lambda: closed_box(2, 9, 13)}.get(name, lambda: closed_box(12, 10, 9))()
        x = {"face": 7, "inner": 5, "sheets": 1, "iolets": 7}[name]
        _cut(g, _plane(x, (INLET, INLET) if name == "iolets" else (WALL, WALL)), rng)
    else:  # random links of every direction
        g = sparse_blob(20, spheres=3) if name == "blob" else closed_box(11, 10, 12)
        some = {"blob": [(WALL, WALL)]}.get(name, [(WALL, WALL), (INLET, INLET), (WALL, INLET), (INLET, WALL)])
        made = _cut(g, lambda *a: some[rng.integers(len(some))] if rng.uniform() < 0.15 else None, rng)
        assert {e for e, _ in made} == set(range(1, 19))
        if name == "ladd":
            kind, bc = IoletSpec(H.PARABOLIC, (6.0, 5.0, 6.0), (1, 0, 0), radius=20.0, max_speed=0.02), H.IOLET_LADD
    if name in ("mixed", "ladd"):  # an iolet link opposite a wall link, on either side of q = 1/2
        wall, io = g.link_type == WALL, (g.link_type == INLET)[:, INV[1:] - 1]
        assert (wall & io & (g.link_dist >= 0.5)).any() and (wall & io & (g.link_dist < 0.5)).any()
    wall = g.link_type == WALL
    g.link_dist[wall] = rng.choice(DIST, int(wall.sum()))
    inlets = [kind] if (g.link_type == INLET).any() else []
    return Case(g, kernel=H.KERNEL_TRT, wall_bc=wall_bc, inlet_bc=bc, tau=0.7, inlets=inlets, outlets=outlets)


def _f0(n):
    return W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))


NAMES = ["face", "inner", "sheets", "cube", "blob", "iolets", "mixed", "ladd"]


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("wall_bc", [H.WALL_SBB, H.WALL_BFL, H.WALL_GZS])
@pytest.mark.parametrize("name", NAMES)
def test_fp64_bitwise(name, wall_bc, general, monkeypatch):
    if wall_bc == H.WALL_GZS and name not in ("face", "blob", "mixed", "ladd"):
        pytest.skip("one plain and the random septa serve for GZS")
    if general:
        monkeypatch.setenv("HLB_FP64_GENERAL_GATHER", "1")
    case = _case(name, wall_bc)
    lat, ref = case.product(), case.oracle()
    f0 = _f0(case.geom.n_sites)
    lat.upload_f(f0, 1)
    ref.set_f(f0, 1)
    for steps in (1, 2, 3):  # each ends in a property step; the next starts from its state
        lat.step(steps, properties=True)
        ref.run(steps, properties=True)
        assert np.array_equal(lat.download_f(), ref.f())
        for got, want in zip(lat.fields(), ref.fields()):
            assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("name", ["face", "mixed"])
def test_neighbour_tables(name):
    """The table from the device names the site itself for such links, as the host's does."""
    case = _case(name, H.WALL_BFL)
    lat = case.product()
    push, pull = lat.neighbour_tables()
    lat.init_equilibrium(1.0)
    dpush, dpull = lat.neighbour_tables()
    assert np.array_equal(push, dpush) and np.array_equal(pull, dpull)


@pytest.mark.parametrize("wall_bc", [H.WALL_SBB, H.WALL_BFL])
@pytest.mark.parametrize("name", NAMES)
def test_fp32(name, wall_bc):
    case = _case(name, wall_bc)
    f0 = _f0(case.geom.n_sites)
    ref = case.oracle()
    ref.set_f(f0, 1)
    ref.run(6, properties=True)
    seen = []
    for variant in (None, 36 + 1):  # one and two slabs per wavefront
        lat = case.product(precision=H.FP32_SHIFTED)
        if variant is not None:
            lat.set_variant(variant)
        lat.upload_f(f0, 1)
        lat.step(4)
        lat.step(2, properties=True)
        seen.append(lat.download_f())
    plain = Case(closed_box(9, 9, 9), kernel=H.KERNEL_LBGK, tau=0.8).product(precision=H.FP32_SHIFTED)
    plain.init_equilibrium(1.0)
    member = case.product(precision=H.FP32_SHIFTED)
    member.upload_f(f0, 1)
    batch = H.Batch([plain, member])
    batch.step(6, properties=True)
    seen.append(member.download_f())
    batch.close()
    assert np.array_equal(seen[0], seen[1]) and np.array_equal(seen[0], seen[2])
    # deviations from w of a few 1e-2 w, six steps of a few dozen roundings each
    assert np.abs(seen[0] - ref.f()).max() <= 6 * 40 * 2.0 ** -24 * 0.05
