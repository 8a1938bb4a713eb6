"""Sequences long enough to be replayed from captured graphs (16 steps and more on
small lattices): from rest, with and without properties, of odd and even lengths
(both buffer parities) and repeated, timed, across a 1024-step chunk, beyond the
number of graphs kept, and after a change of tau, which the captured FP64 launches
hold; eager work and read-backs in between.  The same bits as launched step by step
and, in FP64, as the oracle."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import bifurcation_case, windkessel_cylinder_case

pytestmark = pytest.mark.gpu


def _equal(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))


@pytest.mark.parametrize("precision", [H.FP64, H.FP32_SHIFTED])
def test_replays_match_eager_launches(precision):
    case = bifurcation_case(rp=8.0, lp=40.0, rd=6.5, ld=32.0, steps=3000, peak=0.03, period=200.0)
    lats = [case.product(precision=precision) for _ in range(2)]
    ref = case.oracle() if precision == H.FP64 else None
    for lat, graphs in zip(lats, (True, False)):
        lat.set_graphs(graphs)
    for s in lats + [r for r in (ref,) if r]:
        s.init_equilibrium(1.0)

    def go(n, properties=False, timed=False):
        for lat in lats:
            lat.step_timed(n, properties=properties) if timed else lat.step(n, properties=properties)
        if ref:
            ref.run(n, properties=properties, threads=0)

    def check(held):
        state = [(lat.download_f(), *lat.fields()) for lat in lats]
        assert _equal(*state)
        if ref:
            assert np.array_equal(state[0][0], ref.f()) and _equal(state[0][1:], ref.fields())
        assert [lat.captured_graphs() for lat in lats] == [held, 0]

    go(17)  # the first step gathers nothing
    go(16, properties=True)
    check(2)
    go(17, properties=True)
    check(3)
    go(2)
    for _ in range(3):  # 35 steps a round: each length in both parities
        go(17)
        go(18, timed=True)
    go(1, properties=True)
    check(3 + 2 * 2 if ref else 3 + 1)  # FP64 graphs are kept per buffer parity and first step
    go(1024 + 16)
    go(3, properties=True)
    check(8 if ref else 3 + 1 + 2)
    for n in range(20, 31):  # more than are kept
        go(n)
    go(18)
    go(3, properties=True)
    check(8)
    for tau in (0.62, 0.58):
        for s in lats:
            p = s.get_params()
            p.tau = tau
            s.set_params(p)
            assert s.captured_graphs() == 0
        if ref:
            break
        go(16, properties=True)
        check(1)
    if ref:  # the oracle's tau is fixed: a second one takes the state over
        case.tau = 0.62
        again = case.oracle()
        again.set_f(lats[0].download_f(), lats[0].timestep())
        for k in range(3):
            for lat in lats:
                lat.step(17, properties=True)
            again.run(17, properties=True, threads=0)
            state = [(lat.download_f(), *lat.fields()) for lat in lats]
            assert _equal(*state) and np.array_equal(state[0][0], again.f()) and _equal(state[0][1:], again.fields())
        assert lats[0].captured_graphs() == 2 and lats[1].captured_graphs() == 0
    assert lats[0].timestep() == lats[1].timestep()


CALLS = (16, 17, 1, 33, 16, 2, 17, 33, 16)


@pytest.mark.parametrize("kind,radius", [(H.WK2, 3.0), (H.WK3, 4.6), (H.WK2, 10.5)])
def test_windkessel_state_after_replays(kind, radius):
    case = windkessel_cylinder_case(kind=kind, radius=radius, length=17, box_xy=24)
    lat, ref = case.product(), case.oracle()
    lat.init_equilibrium(1.0)
    ref.init_equilibrium(1.0)
    for n in CALLS + CALLS:
        lat.step(n, properties=n == 33)
        ref.run(n, properties=n == 33)
        assert np.array_equal(lat.iolet_state(True, 0), ref.iolet_state(True, 0))
    assert np.array_equal(lat.download_f(), ref.f())
    assert lat.captured_graphs() >= 4


def test_windkessel_fp32_replayed_eager_and_batched():
    cases = [windkessel_cylinder_case(kind=k, radius=r, length=17, box_xy=24)
             for k, r in ((H.WK2, 3.0), (H.WK3, 6.0), (H.WK3, 10.5))]

    def made():
        lats = [c.product(precision=H.FP32_SHIFTED) for c in cases]
        for lat in lats:
            lat.init_equilibrium(1.0)
        return lats

    replayed, eager, members = made(), made(), made()
    batch = H.Batch(members)
    for lat in eager:
        lat.set_graphs(False)
    for n in CALLS + CALLS:
        for lat in replayed + eager:
            lat.step(n)
        batch.step(n)
        for a, b, c in zip(replayed, eager, members):
            assert np.array_equal(a.iolet_state(True, 0), b.iolet_state(True, 0))
            assert np.array_equal(a.iolet_state(True, 0), c.iolet_state(True, 0))
    for a, b, c in zip(replayed, eager, members):
        assert np.array_equal(a.download_f(), b.download_f()) and np.array_equal(a.download_f(), c.download_f())
        assert a.captured_graphs() == 3 and b.captured_graphs() == 0
    assert batch.captured_graphs() == 3
    batch.close()


@pytest.mark.parametrize("precision", [H.FP64, H.FP32_SHIFTED])
def test_autotuner_times_what_a_solve_runs(precision):
    """Trials of a small lattice are replays, whatever their length, as its solve's
    sequences are; launched eagerly where graphs are off."""
    case = windkessel_cylinder_case(radius=4.6, length=17, box_xy=24)
    for graphs in (True, False):
        lat = case.product(precision=precision)
        lat.set_graphs(graphs)
        lat.init_equilibrium(1.0)
        lat.autotune(3)
        assert lat.captured_graphs() == (8 if graphs else 0)
        lat.step_timed(3)  # times what step(3) runs
        assert lat.captured_graphs() == (8 if graphs else 0)
    if precision == H.FP32_SHIFTED:
        for graphs in (True, False):
            members = [case.product(precision=precision) for _ in range(2)]
            for lat in members:
                lat.init_equilibrium(1.0)
            batch = H.Batch(members)
            batch.set_graphs(graphs)
            batch.autotune(3)
            assert batch.captured_graphs() == (1 if graphs else 0)  # the last variant's
            batch.close()
