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
