"""Currents that travel with a one-step call's launch, held by the lanes of every
wavefront: the same bits as the three-sweep steps, for workgroups of fewer
threads than sources, several planes and rows per tile, and the largest list."""
import numpy as np
import pytest

from fdtd_method_amd import FDTD, Parameters, Precision

pytestmark = pytest.mark.gpu

C = 3e10


@pytest.mark.parametrize("prec", [Precision.FP64, Precision.FP32])
@pytest.mark.parametrize("shape,count,tuning", [
    ((3, 2, 4), 32, (1, 1, 1)),        # 6 threads would hold 6 of 32 sources
    ((5, 4, 3), 32, None),
    ((17, 9, 6), 31, (1, 4, 6)),       # every plane in one tile; a last tile of one row
    ((64, 5, 7), 32, (2, 1, 3)),
    ((48, 40, 20), 1, None),
])
def test_launch_currents(prec, shape, count, tuning):
    dt = 0.5 / (C * np.sqrt(3.0))
    n = int(np.prod(shape))
    rng = np.random.default_rng(11)
    state = [rng.standard_normal(n) * 1e-3 for _ in range(6)]
    a, b = (FDTD(Parameters(*shape, dx=1.0, dy=1.0, dz=1.0), dt, prec) for _ in range(2))
    for g in (a, b):
        for c in range(6):
            g.upload(c, state[c])
    if tuning:
        b.set_tuning(*tuning)
    keys = rng.choice(3 * n, count, replace=False)
    for _ in range(4):
        v = rng.standard_normal(count) / dt
        for g in (a, b):
            g.set_current_values(keys // 3, 6 + keys % 3, v)
        a.update_fields_3sweep(1)
        b.update_fields(1)
        assert a.checksum() == b.checksum()
    a.close()
    b.close()


@pytest.mark.parametrize("prec,shape,count,tuning", [
    (Precision.FP16, (3, 2, 4), 32, (1, 1, 1)),
    (Precision.FP16, (16, 5, 7), 32, (4, 2, 3)),    # 12 lanes of four cells hold cells, 32 hold sources
    (Precision.FP16, (48, 40, 20), 7, None),
    (Precision.FP32, (8, 6, 5), 32, (4, 2, 2)),     # 6 lanes
    (Precision.FP32, (12, 3, 64), 29, (2, 2, 5)),
    (Precision.FP64, (8, 6, 5), 32, (4, 1, 2)),     # 4 lanes
    (Precision.FP64, (10, 7, 3), 30, (2, 3, 3)),    # a last tile of one row
])
def test_sources_held_by_lanes_without_cells(prec, shape, count, tuning):
    """Wide lanes and wavefronts most of whose lanes work on no cell: the same
    bits as the same values as point sources, which take the list, in every
    precision."""
    dt = 0.5 / (C * np.sqrt(3.0))
    n = int(np.prod(shape))
    rng = np.random.default_rng(12)
    state = [rng.standard_normal(n) * 1e-3 for _ in range(6)]
    a, b = (FDTD(Parameters(*shape, dx=1.0, dy=1.0, dz=1.0), dt, prec) for _ in range(2))
    keys = rng.choice(3 * n, count, replace=False)
    for g in (a, b):
        for c in range(6):
            g.upload(c, state[c])
        if tuning:
            g.set_tuning(*tuning)
    for _ in range(4):
        v = rng.standard_normal(count) / dt
        b.set_current_values(keys // 3, 6 + keys % 3, v)
        b.update_fields(1)
        a.set_point_sources([dict(i=int(k // 3 % shape[0]), j=int(k // 3 // shape[0] % shape[1]),
                                  k=int(k // 3 // shape[0] // shape[1]), comp=int(k % 3), kind=0,
                                  amp=float(x)) for k, x in zip(keys, v)])
        a.update_fields(1)
        assert a.checksum() == b.checksum()
    a.close()
    b.close()
