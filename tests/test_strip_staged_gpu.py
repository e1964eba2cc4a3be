"""Strip passes whose planes go through LDS (rows of whole 16-byte packs) and
the direct path beside them (any other row length).

Tile edges: rows of one pack, the last column of a tile and the first of the
next, a tile short of a pack, rows shorter than a tile (the window wraps
several times), one-plane grids, odd and even wavefront counts, z chunks of
one plane, several calls (each call's first pass takes the B half step itself,
and may be its last) and sources in the first
and last cells of tiles.  Every run must equal unblocked single sweeps bit
for bit, in E, B and the probes.
"""
import numpy as np
import pytest

from conftest import courant_dt, random_state
from fdtd_method_amd import FDTD, Parameters, Precision
from fdtd_method_amd.batch import Batch

pytestmark = pytest.mark.gpu

FP64, FP32, FP16 = Precision.FP64, Precision.FP32, Precision.FP16


def make(shape, prec, seed, sources=True):
    dt = courant_dt(1, 1, 1, factor=0.5)
    g = FDTD(Parameters(*shape), dt, prec)
    for c, v in enumerate(random_state(int(np.prod(shape)), seed)):
        g.upload(c, v)
    if sources:
        Ni, Nj, Nk = shape
        g.set_point_sources([dict(i=i % Ni, j=j % Nj, k=k % Nk, comp=q % 3, kind=0, amp=0.3 / dt)
                             for q, (i, j, k) in enumerate([(0, 0, 0), (47, 23, 1), (48, 24, 0),
                                                            (23, 8, 2), (24, -1, -1), (-1, 7, 3)])])
    return g


@pytest.mark.parametrize("prec,shape,L,W,kchunk", [
    (FP32, (4, 3, 1), 4, 16, 0),      # one pack per row, one plane
    (FP32, (48, 24, 9), 4, 16, 0),    # exactly one tile
    (FP32, (52, 25, 9), 4, 16, 1),    # one pack and one row more, chunks of one plane
    (FP32, (100, 30, 12), 3, 8, 5),
    (FP32, (96, 50, 7), 2, 4, 0),
    (FP32, (64, 20, 8), 4, 9, 0),     # odd wavefront count: direct
    (FP32, (51, 26, 9), 4, 16, 0),    # rows that are no whole packs: direct
    (FP64, (2, 5, 3), 4, 8, 0),
    (FP64, (24, 24, 9), 4, 8, 0),
    (FP64, (50, 49, 10), 3, 8, 4),
    (FP64, (26, 26, 6), 2, 4, 1),
    (FP64, (33, 25, 9), 4, 8, 0),     # direct
    (FP16, (8, 9, 2), 4, 16, 0),
    (FP16, (56, 24, 9), 4, 16, 0),
    (FP16, (64, 25, 11), 3, 16, 4),
    (FP16, (60, 24, 9), 4, 16, 0),    # direct
])
def test_strip_planes_through_lds(prec, shape, L, W, kchunk):
    a, b = make(shape, prec, 7), make(shape, prec, 7)
    a.set_time_blocking_strips(0)
    b.set_time_blocking_strips(L, 1, 2, W, kchunk)
    Ni, Nj, Nk = shape
    cells = [(0, 0, 0, 0), (Ni - 1, Nj - 1, Nk - 1, 5), (min(47, Ni - 1), min(23, Nj - 1), 0, 4),
             (min(48, Ni - 1), 0, Nk // 2, 2)]
    for probes in (False, True):
        for g in (a, b):
            if probes:
                g.set_probes(cells, 4 * L + 1)
        for n in (2 * L, L + 1, L):
            a.update_fields(n)
            b.update_fields(n)
            assert a.checksum() == b.checksum(), (probes, n)
    assert np.array_equal(a.read_probes(), b.read_probes())
    assert b.launch_stats()["passes"] > 0


@pytest.mark.parametrize("prec", [FP64, FP32, FP16])
@pytest.mark.parametrize("sides", [((48, 24, 8), (112, 26, 5), (160, 9, 12), (16, 50, 3)),
                                   ((48, 24, 8), (51, 26, 5))])
def test_batch_strips_through_lds(prec, sides):
    a = [make(s, prec, 3 + q) for q, s in enumerate(sides)]
    b = [make(s, prec, 3 + q) for q, s in enumerate(sides)]
    batch = Batch(b)
    batch.set_time_blocking_strips(4, 1, 2, 8 if prec == FP64 else 16)
    for g in a:
        g.set_time_blocking_strips(0)
        g.set_step_carry(False)  # a batch call starts from the B/2 prologue
    for n in (8, 5, 4):
        for g in a:
            g.update_fields(n)
        batch.update_fields(n)
        assert [g.checksum() for g in a] == [g.checksum() for g in b], n
