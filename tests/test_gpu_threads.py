"""Lattices made, stepped (in sequences that are captured and replayed), read back and
dropped by several threads at once, and one that steps throughout: nothing fails, and
every result has the bits of the same work done alone."""
import threading

import numpy as np
import pytest

import hemepure_amd as H
from fixtures import cylinder_case, stenosis_case, windkessel_cylinder_case

pytestmark = pytest.mark.gpu


def _one(case, precision):
    lat = case.product(precision=precision)
    lat.init_equilibrium(1.0)
    lat.step(30, properties=True)
    lat.step(17)
    out = (lat.download_f(), *lat.fields(), lat.iolet_state(True, 0))
    mon = lat.monitor()
    lat.close()
    return out, mon


def _same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a[0], b[0])) and a[1] == b[1]


@pytest.mark.parametrize("threads", [2, 8])
def test_many_threads(threads):
    cases = [stenosis_case(6.0, 40), windkessel_cylinder_case(radius=6.0, length=20),
             cylinder_case(radius=5.0, length=30, box_xy=16), windkessel_cylinder_case(kind=H.WK2, radius=4.6, length=17)]
    work = [(c, p) for c in cases for p in (H.FP64, H.FP32_SHIFTED)]
    want = [_one(*w) for w in work]
    failures = []

    def run(t):
        try:
            for k in range(6):
                i = (t + 3 * k) % len(work)
                assert _same(_one(*work[i]), want[i]), f"thread {t} work {i}"
        except Exception as e:  # noqa: BLE001 - reported below
            failures.append(repr(e))

    pool = [threading.Thread(target=run, args=(t,)) for t in range(threads)]
    for t in pool:
        t.start()
    members = [c.product(precision=H.FP32_SHIFTED) for c in cases]
    for m in members:
        m.init_equilibrium(1.0)
    batch = H.Batch(members)
    for n in (16, 17, 30, 16, 17):
        batch.step(n, properties=True)
    for t in pool:
        t.join()
    assert not failures, failures[:3]
    alone = cases[1].product(precision=H.FP32_SHIFTED)
    alone.init_equilibrium(1.0)
    alone.step(96, properties=True)
    assert np.array_equal(members[1].download_f(), alone.download_f())
    batch.close()
