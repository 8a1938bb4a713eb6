"""Windkessel state over sequences of steps: the sum of one step's flux terms is
taken by the next step's launch (or by the end of the sequence), so calls of
every length, odd and even, eager and replayed, alone and in a batch, must
leave the state the reference has between steps.  Outlets below, at and beyond
one wavefront's 64 coupling sites."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import windkessel_cylinder_case

pytestmark = pytest.mark.gpu

CALLS = (1, 1, 2, 3, 1, 4, 1, 7)


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("kind,radius", [(H.WK2, 3.0), (H.WK3, 4.6), (H.WK3, 6.0), (H.WK2, 10.5)])
def test_fp64_state_after_every_call(kind, radius, graphs):
    case = windkessel_cylinder_case(kind=kind, radius=radius, length=17, box_xy=24)
    lat, ref = case.product(), case.oracle()
    lat.set_graphs(graphs)
    lat.init_equilibrium(1.0)
    ref.init_equilibrium(1.0)
    for n in CALLS + CALLS:
        lat.step(n, properties=n == 3)
        ref.run(n, properties=n == 3)
        assert np.array_equal(lat.iolet_state(True, 0), ref.iolet_state(True, 0))
    assert np.array_equal(lat.download_f(), ref.f())
    assert lat.step_timed(0) >= 0.0
    assert np.array_equal(lat.iolet_state(True, 0), ref.iolet_state(True, 0))


def test_fp32_calls_split_anyhow_and_batched_give_the_same_bits():
    cases = [windkessel_cylinder_case(kind=k, radius=r, length=17, box_xy=24)
             for k, r in ((H.WK2, 3.0), (H.WK3, 6.0), (H.WK3, 10.5))]
    total = sum(CALLS)

    def end(lats, step):
        for lat in lats:
            lat.init_equilibrium(1.0)
        step()
        return [(lat.iolet_state(True, 0), lat.download_f()) for lat in lats]

    whole = [c.product(precision=H.FP32_SHIFTED) for c in cases]
    want = end(whole, lambda: [lat.step(total) for lat in whole])
    parts = [c.product(precision=H.FP32_SHIFTED) for c in cases]
    got = end(parts, lambda: [lat.step(n) for lat in parts for n in CALLS])
    members = [c.product(precision=H.FP32_SHIFTED) for c in cases]
    batch = H.Batch(members)
    together = end(members, lambda: [batch.step(n) for n in CALLS])
    batch.close()
    for a, b, c in zip(want, got, together):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        assert np.array_equal(a[0], c[0]) and np.array_equal(a[1], c[1])
