"""The Windkessel flux sums at every remainder of their loops -- one lane, one row of
16, one load of 64, the loads taken ahead, the tree's rounds of 1024 -- against the
oracle, bitwise in FP64; the FP32 form's tree split over calls anyhow.  And their
time: the sum rides in the next step's launch, so a wide outlet's step takes no more
than the step and the sum one after the other."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import CZ, Case, IoletSpec, W, closed_box, windkessel_cylinder_case

pytestmark = pytest.mark.gpu

SECTIONS = [(1, 1), (1, 15), (4, 4), (1, 17), (7, 9), (8, 8), (5, 13), (1, 79), (8, 10), (15, 17), (16, 16), (1, 257),
            (16, 20), (31, 33), (32, 32), (25, 41), (35, 37), (37, 36), (32, 64), (41, 50)]


def _duct(nx, ny, kind):
    """A closed box whose z end is a Windkessel outlet: nx ny coupling sites."""
    g = closed_box(nx, ny, 3)
    top = g.coords[:, 2] == 3
    for d in range(1, 19):
        if CZ[d] > 0:
            g.link_type[top, d - 1] = H.LINK_OUTLET
            g.link_iolet[top, d - 1] = 0
    out = IoletSpec(kind, ((nx + 1) / 2, (ny + 1) / 2, 3.5), (0, 0, -1), radius=float(nx + ny), area=float(nx * ny),
                    resistance=0.1, r_c=0.001, r_p=0.1, capacitance=3000.0)
    return Case(g, kernel=H.KERNEL_LBGK, tau=0.8, outlets=[out])


def _f0(n):
    return W * (1.0 + 0.02 * np.random.default_rng(1).uniform(-1.0, 1.0, (n, 19)))


@pytest.mark.parametrize("section", SECTIONS, ids=lambda s: str(s[0] * s[1]))
def test_sums(section):
    case = _duct(*section, H.WK3 if section[0] % 2 else H.WK2)
    f0 = _f0(case.geom.n_sites)
    lat, ref = case.product(), case.oracle()
    lat.upload_f(f0, 1)
    ref.set_f(f0, 1)
    for n in (1, 1, 2, 5):
        lat.step(n)
        ref.run(n)
        assert np.array_equal(lat.iolet_state(True, 0), ref.iolet_state(True, 0))
    assert np.array_equal(lat.download_f(), ref.f())
    whole, parts = (case.product(precision=H.FP32_SHIFTED) for _ in range(2))
    for s in (whole, parts):
        s.upload_f(f0, 1)
    whole.step(9)
    for n in (1, 1, 2, 5):
        parts.step(n)
    assert np.array_equal(whole.iolet_state(True, 0), parts.iolet_state(True, 0))
    want, got = ref.iolet_state(True, 0), whole.iolet_state(True, 0)
    # the flow is a mean of velocities of a few 1e-3, nine steps of a few dozen roundings each of g ~ 0.05
    assert abs(got[2] - want[2]) <= case.outlets[0].area * 9 * 40 * 2.0 ** -24 * 0.05


@pytest.mark.parametrize("precision,radius,terms", [(H.FP64, 60.0, 11300), (H.FP32_SHIFTED, 100.0, 31400)])
def test_a_wide_outlet_costs_no_more_than_step_and_sum_in_turn(precision, radius, terms):
    case = windkessel_cylinder_case(radius=radius, length=24, box_xy=int(2 * radius + 11) // 8 * 8)
    times = []
    for kind in (H.WK3, H.COSINE):
        case.outlets[0].kind = kind
        lat = case.product(precision=precision)
        lat.init_equilibrium(1.0)
        lat.step_timed(200)
        times.append(1e6 * min(lat.step_timed(200) for _ in range(4)) / 200)
        lat.close()
    # what a launch of its own took a term: added in order 7.5 ns, as a tree 0.6 ns
    allowed = (7.5 if precision == H.FP64 else 0.6) * terms
    print(f"[windkessel] {terms} terms: {times[0] / 1e3:.1f} us a step, {times[1] / 1e3:.1f} without")
    assert times[0] <= times[1] + allowed
