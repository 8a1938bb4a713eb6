"""Short calls: monitors, whose result the host polls for, over lattices of one
slab to many workgroups, repeated, with the result's place overwritten in between;
single steps, whose iolet values are read in place, against the same steps in one
sequence and the oracle."""
import numpy as np
import pytest

import hemepure_amd as H
from fixtures import Case, W, closed_box, four_cube, IoletSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 9, 17), (65, 30, 30)])
def test_monitor(dims):
    case = Case(closed_box(*dims), kernel=H.KERNEL_LBGK, tau=0.7)
    lat = case.product()
    rng = np.random.default_rng(3)
    lat.upload_f(W * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, (lat.n, 19))), 1)
    for _ in range(3):
        lat.step(1, properties=True)
        rho, u, _ = lat.fields()
        first = lat.monitor()
        assert lat.stable()
        assert first == lat.monitor() == lat.monitor_noalloc()  # the same bits
        assert first["rho_min"] == rho.min() and first["rho_max"] == rho.max()
        # the root of three rounded squares, and a sum of n values near 1 in another order
        speed = np.sqrt((u * u).sum(1)).max()
        assert abs(first["u_max"] - speed) <= 4 * 2.0 ** -53 * speed
        assert abs(first["mass"] - rho.sum()) <= lat.n * 2.0 ** -53 * rho.sum()


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("inlet_bc", [H.IOLET_NASH, H.IOLET_LADD])
def test_single_steps(inlet_bc, fp32):
    if inlet_bc == H.IOLET_NASH:
        inlet = IoletSpec(H.COSINE, (4.5, 4.5, 0.5), (0, 0, 1), density_mean=1.01, density_amp=5e-3, period=7.0)
    else:
        inlet = IoletSpec(H.PARABOLIC, (4.5, 4.5, 0.5), (0, 0, 1), radius=9.0, max_speed=0.02)
    case = Case(four_cube(9, seed=2), kernel=H.KERNEL_TRT, tau=0.8, inlet_bc=inlet_bc, inlets=[inlet],
                outlets=[IoletSpec(H.COSINE, (4.5, 4.5, 8.5), (0, 0, -1), density_mean=0.99, density_amp=2e-3,
                                   period=5.0)])
    kw = dict(precision=H.FP32_SHIFTED) if fp32 else {}
    one, many, ref = case.product(**kw), case.product(**kw), case.oracle()
    for s in (one, many, ref):
        s.init_equilibrium(1.0)
    for k in range(9):
        one.step(1, properties=True)
        if k == 4:
            one.step(2)  # rows behind the first come from the device's copy
            one.step(1)
    many.step(12, properties=True)
    ref.run(12, properties=True)
    assert np.array_equal(one.download_f(), many.download_f())
    if not fp32:
        assert np.array_equal(one.download_f(), ref.f())


def test_monitor_behind_a_long_queue():
    """The result arrives long after polling for it has ended; the next step may
    not overwrite what the queued ones still read."""
    case = Case(four_cube(18, seed=2), kernel=H.KERNEL_LBGK, tau=0.8,
                inlets=[IoletSpec(H.COSINE, (8.5, 8.5, 0.5), (0, 0, 1), density_mean=1.01, density_amp=5e-3, period=7.0)],
                outlets=[IoletSpec(H.COSINE, (8.5, 8.5, 17.5), (0, 0, -1), density_mean=0.99)])
    lat, ref = case.product(), case.oracle()
    for s in (lat, ref):
        s.init_equilibrium(1.0)
    lat.step(700, properties=True)  # a few ms
    a = lat.monitor()
    lat.step(1, properties=True)
    ref.run(701, properties=True)
    assert np.array_equal(lat.download_f(), ref.f())
    assert lat.monitor() != a
