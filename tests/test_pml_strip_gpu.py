"""PML strip passes (two steps per read and write of the state): the same bits,
splits included, as one-step calls, which take the fused sweep, on shapes
around the tiles' edges."""
import numpy as np
import pytest

from fdtd_method_amd import FDTD_PML, Parameters, Precision

pytestmark = pytest.mark.gpu

FP64, FP32 = Precision.FP64, Precision.FP32
C = 3e10


def make(shape, prec, percent):
    dt = 0.5 / (C * np.sqrt(1.0 + 1.0 / 1.44 + 1.0 / 0.81))
    g = FDTD_PML(Parameters(*shape, dx=1.0, dy=1.2, dz=0.9), dt, percent, prec)
    rng = np.random.default_rng(9)
    for c in range(6):
        g.upload(c, rng.standard_normal(int(np.prod(shape))) * 1e-3)
    g.set_point_sources([
        dict(i=shape[0] // 2, j=shape[1] // 2, k=shape[2] // 2, comp=0, kind=0, amp=0.3 / dt),
        dict(i=0, j=1, k=0, comp=1, kind=0, amp=0.2 / dt),          # in the layer: no effect
        dict(i=shape[0] // 2 - 1, j=shape[1] // 2, k=shape[2] // 2 - 1, comp=2, kind=1,
             amp=1e-3 / dt, period=9 * dt, t0=4 * dt, sigma=6 * dt)])
    return g


@pytest.mark.parametrize("prec,shape,percent", [
    (FP64, (56, 60, 80), 0.2),       # whole tiles
    (FP64, (57, 73, 90), 0.3),       # one column and one row more
    (FP64, (122, 60, 44), 0.13),
    (FP64, (40, 180, 171), 0.2),     # narrower than a tile
    (FP64, (130, 40, 60), 0.5),      # all layer
    (FP32, (48, 96, 120), 0.2),
    (FP32, (65, 97, 161), 0.3),
    (FP32, (200, 90, 33), 0.15),     # tiles of layer, main box and both
    (FP32, (131, 57, 90), 0.05),
    (FP32, (232, 40, 70), 0.13),     # packs of both kinds of cells
    (FP32, (34, 300, 301), 0.03),     # one layer cell on each side in x
])
def test_strip_passes_equal_one_step_calls(prec, shape, percent):
    a, b = make(shape, prec, percent), make(shape, prec, percent)
    for n in (2, 5, 8, 1, 4):
        for _ in range(n):
            a.update_fields(1)
        b.update_fields(n)
        assert a.checksum() == b.checksum(), n
    for q in range(12):
        assert np.array_equal(a.split(q), b.split(q)), q
    assert b.launch_stats()["passes"] == 1 + 2 + 4 + 2
    a.close()
    b.close()


def test_more_steps_than_a_table_of_source_values():
    a, b = make((96, 90, 100), FP32, 0.2), make((96, 90, 100), FP32, 0.2)
    for _ in range(523):
        a.update_fields(1)
    b.update_fields(523)
    assert a.checksum() == b.checksum()
    assert b.launch_stats()["passes"] == 261


@pytest.mark.parametrize("prec", [FP64, FP32])
def test_path_2_runs_every_step_as_a_sweep(prec):
    """set_pml_path(2) turns the passes off, 0 on again: the same bits, and the
    sweeps take the shape that set_tuning gives."""
    a, b = make((96, 90, 100), prec, 0.2), make((96, 90, 100), prec, 0.2)
    passes = 0
    for path, n in ((2, 6), (0, 4), (2, 5), (1, 3), (0, 6), (2, 3), (0, 7), (1, 2)):
        b.set_pml_path(path)
        assert b.get_pml_path()["path"] == path
        if path == 2:
            b.set_tuning(1, 5, 7)
        a.update_fields(n)
        b.update_fields(n)
        assert a.checksum() == b.checksum(), (path, n)
        passes += n // 2 if path == 0 else 0
        assert b.launch_stats()["passes"] == passes
    for q in range(12):
        assert np.array_equal(a.split(q), b.split(q)), q
    with pytest.raises(Exception):
        b.set_pml_path(3)
    a.close()
    b.close()


@pytest.mark.torch
def test_memory_of_the_passes_is_given_back():
    """A grid whose memory is short gives up the passes' second set of B splits,
    with the state in either set, rather than refuse: a record buffer that
    fits only without it is allocated, the runs go on as sweeps with the same
    bits, and passes come back when asked for."""
    import torch

    shape = (256, 256, 256)
    a, b = make(shape, FP64, 0.2), make(shape, FP64, 0.2)
    a.set_pml_path(2)
    a.update_fields(6)
    b.update_fields(6)
    assert b.launch_stats()["passes"] == 3
    free = torch.cuda.mem_get_info()[0]
    b.set_energy_interval(1 << 30, (free + (600 << 20)) // 48)  # of the 768 MiB of that set
    b.set_energy_interval(0)
    assert a.checksum() == b.checksum()
    for q in range(12):
        assert np.array_equal(a.split(q), b.split(q)), q
    a.update_fields(3)
    b.update_fields(3)
    assert a.checksum() == b.checksum()
    assert b.launch_stats()["passes"] == 3
    # a request that no release could meet is refused and costs nothing
    b.set_pml_path(0)
    with pytest.raises(Exception):
        b.set_energy_interval(1 << 30, 1 << 40)
    b.set_energy_interval(0)
    a.update_fields(5)
    b.update_fields(5)
    assert a.checksum() == b.checksum()
    assert b.launch_stats()["passes"] == 5
    a.close()
    b.close()


def test_passes_of_large_grids_march_short_chunks():
    """A pass whose tiles all march the whole grid lets neighbours drift apart
    (512^3 FP32: 4.4 ms against 3.4, two sweeps 6.4)."""
    dt = 0.5 / (C * np.sqrt(3.0))
    g = FDTD_PML(Parameters(512, 512, 512, dx=1.0, dy=1.0, dz=1.0), dt, 0.2, FP32)
    ms = {}
    for path in (2, 0):
        g.set_pml_path(path)
        g.update_fields(4)
        runs = [g.time_update_fields_kernels(12)["steady"] for _ in range(4)]
        ms[path] = min(t / count for t, count in runs)
    assert ms[0] < 0.62 * 2 * ms[2], ms
    g.close()


@pytest.mark.parametrize("prec,side,percent,passes", [
    (FP32, 72, 0.1, False),    # the caches hold the state, packs of both kinds of cells
    (FP64, 72, 0.3, False),    # packs of both kinds
    (FP32, 100, 0.3, False),
    (FP32, 80, 0.1, True), (FP64, 80, 0.3, True), (FP32, 128, 0.1, True),
])
def test_grids_that_take_passes(prec, side, percent, passes):
    """Passes run where they are the faster form, and only there (72^3 FP32: a
    pass 40 us, its two sweeps 27)."""
    a, b = make((side,) * 3, prec, percent), make((side,) * 3, prec, percent)
    a.set_pml_path(2)
    for n in (4, 7):
        a.update_fields(n)
        b.update_fields(n)
        assert a.checksum() == b.checksum()
    assert b.launch_stats()["passes"] == (5 if passes else 0)
    a.close()
    b.close()


@pytest.mark.parametrize("prec,side", [(FP32, 24), (FP32, 64), (Precision.FP16, 40)])
def test_sweeps_with_and_without_the_layers_totals(prec, side):
    """Sweeps that leave out the layer's E totals between the steps of a run,
    or not, by the size of the state: after a run every layer total is the sum
    of its splits, and two such runs agree bit for bit."""
    a, b = make((side,) * 3, prec, 0.2), make((side,) * 3, prec, 0.2)
    for g in (a, b):
        g.set_pml_path(2)
        g.update_fields(5)
    assert a.checksum() == b.checksum()
    for c, (p, q) in enumerate([("Exy", "Exz"), ("Eyx", "Eyz"), ("Ezx", "Ezy")]):
        e, s = a.download(c), a.split(p) + a.split(q)
        layer = np.ones((side,) * 3, bool)
        w = a.pml_widths
        layer[w[2]:side - w[2], w[1]:side - w[1], w[0]:side - w[0]] = False
        d = np.abs(e - s)[layer.ravel()]
        unit = 2.0 ** (-24 if prec == FP32 else -11)
        assert d.max() <= unit * np.abs(s).max()
    a.close()
    b.close()


def test_fp16_sweeps_of_large_grids():
    """FP16 sweeps leave out the layer's totals on large grids, rescaling ones
    never do: a run of both kinds stays within FP16's 5e-3 (relative L2) of FP32
    on planes inside and across the layer, and its last sweep's layer totals are
    the sums of the splits."""
    n = 348
    dt = 0.5 / (C * np.sqrt(3.0))
    grids = []
    for prec in (FP32, Precision.FP16):
        g = FDTD_PML(Parameters(n, n, n, dx=1.0, dy=1.0, dz=1.0), dt, 0.1, prec)
        g.add_plane_wave([2, 3, 1], 0.7, 0.3, [0.3, -1.0, 0.5])
        if prec == Precision.FP16:
            g.autoscale(10)
            g.set_autoscale_interval(2, 10)
        g.update_fields(7)
        grids.append(g)
    a, b = grids
    for k in (0, 33, 34, 35, n // 2, n - 36, n - 1):
        x = [np.concatenate([g.download_plane(c, k).ravel() for c in range(6)]) for g in grids]
        assert np.linalg.norm(x[1] - x[0]) <= 5e-3 * np.linalg.norm(x[0]), k
    e, s = b.download(0)[:n * n], (b.split("Exy") + b.split("Exz"))[:n * n]  # plane 0: all layer
    assert np.abs(e - s).max() <= 2.0 ** -11 * np.abs(s).max()
    a.close()
    b.close()
