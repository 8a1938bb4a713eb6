"""Iolet values in the site's own post-collision row: sites where a BFL wall link
lies opposite an iolet link on either side of q = 1/2 (there the row keeps the
post-collision value), under cached and non-temporal row stores and one or two
slabs per wavefront.  FP64 against the oracle bitwise, FP32 variants against one
another bitwise and against the oracle within the shifted form's tolerance."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import Case, W, four_cube, IoletSpec

pytestmark = pytest.mark.gpu
OPP = np.array([0] + [k + 1 if k % 2 else k - 1 for k in range(1, 19)])


def _case(side):
    g = four_cube(9, seed=2)
    wall = g.link_type == H.LINK_WALL
    g.link_dist[wall] = np.random.default_rng(5).choice(np.array([0.3, 0.5, 0.9], dtype=np.float32), int(wall.sum()))
    io = g.link_type >= H.LINK_INLET
    opposite = io[:, OPP[1:] - 1]
    assert (wall & opposite & (g.link_dist >= 0.5)).any() and (wall & opposite & (g.link_dist < 0.5)).any()
    assert (wall & ~opposite & (g.link_dist >= 0.5)).any()
    return Case(g, kernel=H.KERNEL_TRT, wall_bc=side, tau=0.8,
                inlets=[IoletSpec(H.COSINE, (4.5, 4.5, 0.5), (0, 0, 1), density_mean=1.01)],
                outlets=[IoletSpec(H.COSINE, (4.5, 4.5, 8.5), (0, 0, -1), density_mean=0.99)])


def _f0(n):
    return W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))


@pytest.mark.parametrize("wall_bc", [H.WALL_SBB, H.WALL_BFL])
@pytest.mark.parametrize("variant", [None, 1, 54 + 1])
def test_fp64_bitwise(wall_bc, variant):
    case = _case(wall_bc)
    lat, ref = case.product(), case.oracle()
    if variant is not None:
        lat.set_variant(variant)
    f0 = _f0(case.geom.n_sites)
    lat.upload_f(f0, 1)
    ref.set_f(f0, 1)
    for steps in (1, 2, 5):
        lat.step(steps, properties=True)
        ref.run(steps, properties=True)
        assert np.array_equal(lat.download_f(), ref.f())
        for got, want in zip(lat.fields(), ref.fields()):
            assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("wall_bc", [H.WALL_SBB, H.WALL_BFL])
def test_fp32_variants(wall_bc):
    case = _case(wall_bc)
    f0 = _f0(case.geom.n_sites)
    ref = case.oracle()
    ref.set_f(f0, 1)
    ref.run(8, properties=True)
    seen = []
    for variant in (None, 36 + 1, 108 + 1, 108 + 36 + 1):
        lat = case.product(precision=H.FP32_SHIFTED)
        if variant is not None:
            lat.set_variant(variant)
        lat.upload_f(f0, 1)
        lat.step(3)
        lat.step(5, properties=True)
        seen.append(lat.download_f())
        assert np.array_equal(seen[0], seen[-1])
    # deviations from w of a few 1e-2 w, eight steps of a few dozen roundings each
    assert np.abs(seen[0] - ref.f()).max() <= 8 * 40 * 2.0 ** -24 * 0.05
