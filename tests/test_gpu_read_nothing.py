"""Reading back none of the arrays still waits for the queued steps."""
import time

import pytest

import hemepure_amd as H
from fixtures import Case, closed_box

pytestmark = pytest.mark.gpu


def test_a_read_of_nothing_waits():
    lat = Case(closed_box(64, 64, 64), kernel=H.KERNEL_LBGK, tau=0.8).product()
    lat.init_equilibrium(1.0)
    lat.step(1000)
    lat.synchronize()
    start = time.perf_counter()
    lat.step(1000)
    lat.synchronize()
    steps = time.perf_counter() - start
    for read in (lambda: H.lib().hlb_get_fields(lat._h, None, None, None),
                 lambda: H.lib().hlb_get_stress(lat._h, *[None] * 6)):
        start = time.perf_counter()
        lat.step(1000)
        assert read() == 0
        assert time.perf_counter() - start > 0.5 * steps
