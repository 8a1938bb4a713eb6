"""Site arrays through the chunked, reordering copies: uploads and downloads
at sizes around a chunk's edge (one chunk of distributions is 6848 sites) and
of several chunks and host threads, two lattices at once from two threads, and
the records against plain numpy of the same values."""
import threading

import numpy as np
import pytest

import hemepure_amd as H
from fixtures import Case, W, closed_box

pytestmark = pytest.mark.gpu

BOXES = [(1, 1, 1), (1, 41, 167), (8, 8, 107), (1, 9, 761), (8, 16, 321), (1, 17, 2417), (16, 81, 107)]


def _state(n, seed):
    return W * (1.0 + 0.05 * np.random.default_rng(seed).uniform(-1.0, 1.0, (n, 19)))


def _stored(f, precision):
    """What the storage form holds of f: double, or float of f - w."""
    return f if precision == H.FP64 else (f - W).astype(np.float32).astype(np.float64) + W


@pytest.mark.parametrize("precision", [H.FP64, H.FP32_SHIFTED])
@pytest.mark.parametrize("box", BOXES)
def test_round_trip_and_records(box, precision):
    case = Case(closed_box(*box), kernel=H.KERNEL_TRT, tau=0.7)
    lat = case.product(precision=precision)
    f = _state(lat.n, 1)
    lat.upload_f(f, 3)
    assert lat.timestep() == 3
    g = lat.download_f()
    assert np.array_equal(g, _stored(f, precision))
    # a step that starts from the uploaded state and reports its moments
    lat.step(1, properties=True)
    rho, u, wss = lat.fields()
    # 19 terms near w, rounded in the storage form's precision
    eps = 19 * (2.0 ** -53 if precision == H.FP64 else 2.0 ** -24)
    c = np.stack([np.asarray(v, float) for v in _vectors()], 1)
    np.testing.assert_allclose(rho, g.sum(1), rtol=0, atol=4 * eps)
    np.testing.assert_allclose(u, (g @ c) / g.sum(1)[:, None], rtol=0, atol=4 * eps)
    assert np.isfinite(wss).all()
    # the pressure on the stress tensor's diagonal: its trace is -3 cs^2 (rho - 1) - tr Pi
    lat.upload_f(_state(lat.n, 1), 3)
    ten = lat.stress()
    assert ten.shape == (lat.n, 17)
    p = (g.sum(1) - 1.0) / 3.0
    vm2 = 0.5 * ((ten[:, 0] - ten[:, 3]) ** 2 + (ten[:, 3] - ten[:, 5]) ** 2 + (ten[:, 5] - ten[:, 0]) ** 2) + \
        3.0 * (ten[:, 1] ** 2 + ten[:, 2] ** 2 + ten[:, 4] ** 2)
    # von Mises from the tensor's own components: same row, same site (terms below 0.1, FP64 arithmetic)
    np.testing.assert_allclose(ten[:, 6] ** 2, vm2, rtol=0, atol=1e-13)
    # normal + tangential projection = traction
    np.testing.assert_allclose(ten[:, 8:11], ten[:, 11:14] + ten[:, 14:17], rtol=0, atol=1e-14)
    assert np.isfinite(p).all()


def _vectors():
    from fixtures import CX, CY, CZ

    return CX, CY, CZ


def test_two_lattices_from_two_threads():
    lats = [Case(closed_box(*b), tau=0.8).product(precision=p)
            for b, p in (((16, 81, 107), H.FP64), ((9, 64, 200), H.FP32_SHIFTED))]
    states = [_state(lat.n, 7 + k) for k, lat in enumerate(lats)]
    got = [[], []]

    def loop(k):
        for _ in range(4):
            lats[k].upload_f(states[k], 1)
            got[k].append(lats[k].download_f())

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, precision in enumerate((H.FP64, H.FP32_SHIFTED)):
        want = _stored(states[k], precision)
        assert len(got[k]) == 4 and all(np.array_equal(g, want) for g in got[k])
