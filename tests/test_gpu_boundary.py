"""Boundary records: wall distances at the edges of BFL's two branches (0, just
below 1/2, 1/2, 1), links with a wall on both sides, on slabs of every fill,
with and without iolets, in steady, property and general-gather steps, against
the oracle: bitwise in FP64, within the shifted form's tolerance in FP32."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import Case, W, bifurcation_case, closed_box, four_cube, sparse_blob, IoletSpec

pytestmark = pytest.mark.gpu

EDGES = np.array([0.0, np.nextafter(np.float32(0.5), np.float32(0)), 0.5, 1.0, 0.25, 0.75], dtype=np.float32)


def _case(name, kernel):
    if name == "cube":
        g = four_cube(10, seed=4)
        io = dict(inlets=[IoletSpec(H.COSINE, (4.5, 4.5, 0.5), (0, 0, 1), density_mean=1.01)],
                  outlets=[IoletSpec(H.COSINE, (4.5, 4.5, 8.5), (0, 0, -1), density_mean=0.99)])
    else:
        g = {"box": lambda: closed_box(9, 17, 8), "sheet": lambda: closed_box(1, 9, 13),
             "line": lambda: closed_box(1, 1, 19), "blob": lambda: sparse_blob(24, spheres=3)}[name]()
        io = {}
    wall = g.link_type == H.LINK_WALL
    g.link_dist[wall] = np.random.default_rng(2).choice(EDGES, int(wall.sum()))
    return Case(g, kernel=kernel, wall_bc=H.WALL_BFL, tau=0.7, **io)


def _ladd():
    return bifurcation_case(rp=7.0, lp=30.0, rd=5.5, ld=24.0, steps=20, peak=0.03, period=16.0)


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("name", ["box", "sheet", "line", "blob", "cube", "ladd"])
def test_fp64_bitwise(name, general, monkeypatch):
    if general:
        monkeypatch.setenv("HLB_FP64_GENERAL_GATHER", "1")
    case = _ladd() if name == "ladd" else _case(name, H.KERNEL_TRT)
    n = case.geom.n_sites
    f0 = W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))
    lat, ref = case.product(), case.oracle()
    lat.upload_f(f0, 1)
    ref.set_f(f0, 1)
    for steps in (1, 2, 3):  # each ends in a property step; the next starts from its state
        lat.step(steps, properties=True)
        ref.run(steps, properties=True)
        assert np.array_equal(lat.download_f(), ref.f())
        for got, want in zip(lat.fields(), ref.fields()):
            assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("name", ["box", "sheet", "line", "blob", "cube", "ladd"])
def test_fp32(name):
    case = _ladd() if name == "ladd" else _case(name, H.KERNEL_TRT)
    n = case.geom.n_sites
    f0 = W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))
    lat, ref = case.product(precision=H.FP32_SHIFTED), case.oracle()
    lat.upload_f(f0, 1)
    ref.set_f(f0, 1)
    lat.step(6, properties=True)
    ref.run(6, properties=True)
    # deviations from w of a few 1e-2 w, six steps of a few dozen roundings each
    err = np.abs(lat.download_f() - ref.f()).max()
    assert err <= 6 * 40 * 2.0 ** -24 * 0.05
