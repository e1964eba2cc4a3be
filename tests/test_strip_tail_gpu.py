"""The strip pass that takes the two or three steps a call's full passes leave:
the same bits as single sweeps, at step counts around whole passes, with
sources, probes and in-run rescaling."""
import numpy as np
import pytest

from fdtd_method_amd import FDTD, Parameters, Precision

pytestmark = pytest.mark.gpu

FP64, FP32, FP16 = Precision.FP64, Precision.FP32, Precision.FP16
C = 3e10


def make(shape, prec):
    dt = 0.5 / (C * np.sqrt(3.0))
    g = FDTD(Parameters(*shape, dx=1.0, dy=1.0, dz=1.0), dt, prec)
    rng = np.random.default_rng(5)
    for c in range(6):
        g.upload(c, rng.standard_normal(int(np.prod(shape))) * 1e-3)
    if prec == FP16:
        g.set_scales([2.0 ** 8] * 6)
    g.set_point_sources([
        dict(i=0, j=0, k=0, comp=0, kind=0, amp=0.3 / dt),
        dict(i=shape[0] - 1, j=shape[1] // 2, k=shape[2] - 1, comp=2, kind=1, amp=1e-3 / dt,
             period=9 * dt, t0=4 * dt, sigma=6 * dt)])
    g.set_probes([(0, 0, 0, c) for c in range(6)] + [(shape[0] - 1, 1, shape[2] - 1, 5)], 700)
    return g


@pytest.mark.parametrize("prec,shape,L,counts", [
    (FP64, (50, 26, 9), 4, (6, 7, 2, 11)),
    (FP64, (33, 25, 9), 4, (6, 7)),         # rows that are no whole packs
    (FP32, (52, 25, 9), 4, (6, 7, 3, 10)),
    (FP32, (51, 26, 9), 3, (5, 8)),
    (FP16, (64, 25, 11), 4, (6, 7, 5)),
    (FP32, (16, 8, 4), 4, (258, 263)),      # past a table of source values
    (FP32, (16, 8, 4), 3, (257, 260)),
])
def test_steps_left_over(prec, shape, L, counts):
    a, b = make(shape, prec), make(shape, prec)
    a.set_time_blocking_strips(0)
    b.set_time_blocking_strips(L, 1, 2, 8)
    for n in counts:
        a.update_fields(n)
        b.update_fields(n)
        assert a.checksum() == b.checksum(), n
    assert np.array_equal(a.read_probes(), b.read_probes())
    assert b.launch_stats()["passes"] == sum(n // L for n in counts)
    a.close()
    b.close()


@pytest.mark.parametrize("prec,shape,blocked", [
    (FP64, (72, 70, 74), True),     # just above the size at which passes pay
    (FP64, (64, 64, 64), False),
    (FP32, (33, 150, 181), True),   # one tile across
    (FP32, (72, 70, 74), False),
    (FP16, (120, 120, 120), False),
    (FP64, (3, 2, 200000), False),  # few tiles, many planes
])
def test_default_of_narrow_grids(prec, shape, blocked):
    a, b = make(shape, prec), make(shape, prec)
    assert (b.get_time_blocking_strips()["L"] == 4) == blocked
    a.set_time_blocking_strips(0)
    for n in (4, 11):
        a.update_fields(n)
        b.update_fields(n)
        assert a.checksum() == b.checksum(), n
    a.close()
    b.close()


@pytest.mark.parametrize("prec,shape,n,sweeps", [
    (FP16, (256, 256, 192), 6, 2),   # beyond the last-level cache: two sweeps
    (FP16, (256, 256, 192), 7, 1),   # three steps: a pass
    (FP16, (128, 128, 64), 6, 1),
    (FP16, (257, 256, 192), 6, 1),   # single-cell lanes
    (FP32, (256, 256, 128), 6, 1),
    (FP64, (256, 128, 128), 6, 1),
])
def test_form_of_the_steps_left_over(prec, shape, n, sweeps):
    a, b = make(shape, prec), make(shape, prec)
    a.set_time_blocking_strips(0)
    for _ in range(2):
        a.update_fields(n)
        b.update_fields(n)
        assert a.checksum() == b.checksum()
    s = b.launch_stats()
    assert (s["passes"], s["sweeps"]) == (2, 2 * sweeps)
    a.close()
    b.close()
