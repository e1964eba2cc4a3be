"""Temporal blocking with the wavefront-strip kernel (strip_sweep).

L fused steps per pass over HBM on tiles of 64*V columns by W*R rows must
give exactly the fields of L unblocked fused sweeps (bit-identical in every
precision, since the per-cell expressions are the same), with point
sources, remainders of n % L steps, several tiles and z chunks, and grids
smaller than a tile (ghost cells wrapping several times).  FP64 is also
held to the oracle.
"""
import numpy as np
import pytest

from conftest import courant_dt, random_state
from fdtd_method_amd import FDTD, Parameters, Precision
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def grid(shape, dt, state, prec, sources=()):
    g = FDTD(Parameters(*shape), dt, prec)
    for c in range(6):
        g.upload(c, state[c])
    if sources:
        g.set_point_sources(list(sources))
    return g


def rel_l2(out, ref):
    num = sum(float(np.sum((a - b) ** 2)) for a, b in zip(out, ref))
    den = sum(float(np.sum(b ** 2)) for b in ref)
    return np.sqrt(num / den)


def sources_for(shape, dt):
    Ni, Nj, Nk = shape
    return [dict(i=3, j=Nj - 1, k=0, comp=2, kind=1, amp=1.0, period=16 * dt, t0=5 * dt,
                 sigma=6 * dt),
            dict(i=Ni - 1, j=0, k=Nk - 1, comp=0, kind=0, amp=0.3),
            dict(i=Ni // 2, j=Nj // 2, k=Nk // 2, comp=1, kind=1, amp=0.5, period=9 * dt,
                 t0=0.0, sigma=0.0)]


CASES = [
    # prec, L, V, R, W, kchunk
    (Precision.FP64, 1, 1, 2, 4, 5),
    (Precision.FP64, 2, 1, 2, 8, 0),
    (Precision.FP64, 3, 1, 2, 6, 7),
    (Precision.FP64, 4, 1, 2, 8, 4),
    (Precision.FP32, 4, 1, 2, 8, 0),
    (Precision.FP32, 1, 2, 2, 3, 0),
    (Precision.FP32, 2, 1, 4, 4, 6),
    (Precision.FP32, 2, 2, 2, 8, 0),
    (Precision.FP32, 3, 1, 4, 3, 0),
    (Precision.FP32, 3, 1, 2, 16, 9),
    (Precision.FP32, 4, 2, 2, 5, 3),
    (Precision.FP32, 4, 1, 4, 4, 0),
    (Precision.FP16, 2, 2, 2, 4, 0),
    (Precision.FP16, 3, 1, 4, 2, 5),
]


@pytest.mark.parametrize("prec,L,V,R,W,kchunk", CASES)
def test_strip_blocking_bit_exact(prec, L, V, R, W, kchunk):
    shape = (40, 36, 22)
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1, factor=0.5)
    st = random_state(n, 40)
    src = sources_for(shape, dt)
    a = grid(shape, dt, st, prec, src)
    b = grid(shape, dt, st, prec, src)
    b.set_time_blocking_strips(L, V, R, W, kchunk)
    cfg = b.get_time_blocking_strips()
    print("strips", cfg, flush=True)
    assert (cfg["L"], cfg["V"], cfg["R"], cfg["W"]) == (L, V, R, W)
    for nsteps in (2 * L + 1, L, 3):
        a.update_fields(nsteps)
        b.update_fields(nsteps)
        assert a.checksum() == b.checksum(), nsteps
    if prec == Precision.FP64:
        r = O.OracleGrid(*shape, 1.0, 1.0, 1.0, dt)
        for c in range(6):
            r.fields()[c][:] = st[c]
        r.run_point_sources(src, 2 * L + 1 + L + 3)
        assert rel_l2(b.fields(), r.E + r.B) <= 1e-12


@pytest.mark.parametrize("shape", [(200, 130, 40), (130, 70, 65)], ids=lambda s: "x".join(map(str, s)))
def test_strip_blocking_many_tiles_and_chunks(shape):
    """Several tiles along x and y (partial last tiles) and z chunks."""
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1)
    st = random_state(n, 41)
    src = sources_for(shape, dt)
    a = grid(shape, dt, st, Precision.FP32, src)
    b = grid(shape, dt, st, Precision.FP32, src)
    b.set_time_blocking_strips(3, 1, 4, 4, 16)
    a.update_fields(7)
    b.update_fields(7)
    assert a.checksum() == b.checksum()
    b.set_time_blocking_strips(2, 2, 2, 8, 0)
    a.update_fields(5)
    b.update_fields(5)
    assert a.checksum() == b.checksum()


@pytest.mark.parametrize("storage", ["wide", "fp16"])
def test_strip_blocking_tiny_grids(storage):
    """Grids smaller than one tile: the x ghost columns and y ghost rows wrap
    several times around the grid (FP32 and FP64, or FP16 storage, whose
    strips read and write through plane buffer resources)."""
    for shape, V in [((4, 3, 5), 2), ((2, 2, 2), 2), ((6, 1, 3), 1), ((1, 5, 4), 1)]:
        n = int(np.prod(shape))
        dt = courant_dt(1, 1, 1)
        st = random_state(n, 42)
        if storage == "fp16":
            prec = Precision.FP16
            st = [x * 0.25 for x in st]
        else:
            prec = Precision.FP32 if V == 2 else Precision.FP64  # FP64 strips: V = 1
        a = grid(shape, dt, st, prec)
        b = grid(shape, dt, st, prec)
        b.set_time_blocking_strips(2, V, 2, 4, 1)
        a.update_fields(6)
        b.update_fields(6)
        assert a.checksum() == b.checksum(), shape


def test_strip_blocking_many_sources_on_one_plane():
    """Point sources sorted by plane: many on one plane and on the wrapped
    planes of a chunk's ghost range."""
    shape = (48, 40, 24)
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1)
    st = random_state(n, 43)
    rng = np.random.default_rng(7)
    src = [dict(i=int(rng.integers(48)), j=int(rng.integers(40)), k=k, comp=int(rng.integers(3)),
                kind=1, amp=float(rng.uniform(0.1, 1)), period=float(rng.uniform(8, 30)) * dt,
                t0=0.0, sigma=0.0)
           for k in [0] * 20 + [23] * 5 + [7, 8, 9, 12]]
    a = grid(shape, dt, st, Precision.FP32, src)
    b = grid(shape, dt, st, Precision.FP32, src)
    b.set_time_blocking_strips(4, 1, 2, 8, 6)
    a.update_fields(9)
    b.update_fields(9)
    assert a.checksum() == b.checksum()


def test_strip_blocking_rejects_invalid_shapes():
    shape = (33, 20, 10)
    dt = courant_dt(1, 1, 1)
    g = grid(shape, dt, random_state(int(np.prod(shape)), 44), Precision.FP64)
    for args in [(2, 2, 2, 4, 0),    # V=2 with odd Ni
                 (2, 1, 4, 4, 0),    # FP64 builds V*R*8 <= 16 only
                 (2, 1, 3, 4, 0),    # R not built
                 (5, 1, 2, 4, 0),    # L > 4
                 (2, 1, 2, 1, 0),    # W*R - 2L < 1
                 (2, 1, 2, 17, 0)]:  # W > 16
        with pytest.raises(RuntimeError):
            g.set_time_blocking_strips(*args)
    g.set_time_blocking_strips(0)
    assert g.get_time_blocking_strips()["L"] == 0


@pytest.mark.parametrize("L,V,lanes,TYg", [(2, 2, 32, 12), (3, 1, 64, 8)])
def test_patch_blocking_fp16_bit_exact(L, V, lanes, TYg):
    """The ghost-zone patch kernel with FP16 storage: every level's fields
    are rounded to FP16 as between unblocked sweeps."""
    shape = (40, 36, 22)
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1, factor=0.5)
    st = random_state(n, 45)
    src = sources_for(shape, dt)
    a = grid(shape, dt, st, Precision.FP16, src)
    b = grid(shape, dt, st, Precision.FP16, src)
    # patch passes start every call from the B/2 prologue (no carried half
    # step): compare with unblocked calls that do the same
    a.set_step_carry(False)
    b.set_time_blocking(L, V, lanes, TYg, 0)
    for nsteps in (2 * L + 1, L, 3):
        a.update_fields(nsteps)
        b.update_fields(nsteps)
        assert a.checksum() == b.checksum(), nsteps


@pytest.mark.parametrize("prec", [Precision.FP16, Precision.FP32])
def test_strip_blocking_carries_the_half_step(prec):
    """Strip runs carry the next half step across calls like the unblocked
    path: calls of L steps (and of L+1: a pass plus a fused remainder)
    equal one long unblocked call bitwise, FP16 included."""
    shape = (64, 40, 18)
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1)
    st = [x * 0.25 for x in random_state(n, 46)]
    src = sources_for(shape, dt)
    a = grid(shape, dt, st, prec, src)
    b = grid(shape, dt, st, prec, src)
    b.set_time_blocking_strips(3, 1, 2, 8, 0)
    for nsteps in (3, 3, 4, 3):
        b.update_fields(nsteps)
    a.update_fields(13)
    assert a.checksum() == b.checksum()


@pytest.mark.parametrize("kind", ["strips", "patch"])
def test_blocking_with_dense_currents_runs_single_sweeps(kind):
    """A dense J array (a whole J component uploaded) is read by single
    sweeps: with blocking set, such runs still equal unblocked ones, and
    blocking resumes once the dense J is dropped."""
    shape = (32, 20, 12)
    n = int(np.prod(shape))
    dt = courant_dt(1, 1, 1)
    st = random_state(n, 47)
    J = np.random.default_rng(5).standard_normal(n) * 1e-3
    a = grid(shape, dt, st, Precision.FP64)
    b = grid(shape, dt, st, Precision.FP64)
    if kind == "strips":
        b.set_time_blocking_strips(2, 1, 2, 8, 0)
    else:
        b.set_time_blocking(2, 1, 32, 12, 0)
    for g in (a, b):
        g.upload(7, J)  # dense JY
        g.update_fields(5)
    assert a.checksum() == b.checksum()
    for g in (a, b):
        g.zeroed_currents()
        g.update_fields(4)
    assert a.checksum() == b.checksum()


def test_strip_blocking_fp16_in_run_rescaling():
    """FP16 strip passes with in-run rescaling (a decision every 8 steps, two
    passes of L=4): a blocked run rescales the state in place between
    passes, where an unblocked run scales a sweep's output, so the two agree
    to FP16 rounding rather than bitwise.  The scales follow a growing
    point-source field, and the result stays within 5e-3 of FP64 and close to
    the unblocked rescaling run."""
    N = 40
    dt = courant_dt(1, 1, 1, factor=0.5)
    src = [dict(i=20, j=20, k=20, comp=2, kind=1, amp=1.0, period=20 * dt, t0=60 * dt,
                sigma=20 * dt)]

    def make(prec, blocking):
        g = FDTD(Parameters(N, N, N), dt, prec)
        g.set_point_sources(src)
        if prec == Precision.FP16:
            g.autoscale(target_log2=10, magnitude_floor=4.0 * np.pi * dt * 1e-2)
            g.set_autoscale_interval(8, 10)
        if blocking:
            g.set_time_blocking_strips(*blocking)
        return g

    ref = make(Precision.FP64, None)
    ub = make(Precision.FP16, None)
    bl = make(Precision.FP16, (4, 1, 2, 8, 0))
    s0 = bl.get_scales()
    for g in (ref, ub, bl):
        g.update_fields(90)
    s1 = bl.get_scales()
    assert s1 != s0
    mx = bl.max_abs()
    for c in (0, 1, 2, 3, 4):  # Bz stays ~0 under a Jz source
        assert 2.0 ** 6 <= mx[c] * s1[c] <= 2.0 ** 14, (c, mx[c] * s1[c])

    err = bl.compare(ref)
    r_ref = np.sqrt(sum(e[0] for e in err) / sum(e[1] for e in err))
    r_ub = rel_l2(bl.fields(), ub.fields())
    print("fp16 blocked rescaling: relL2 vs FP64", r_ref, "vs unblocked FP16", r_ub, s0, s1)
    assert r_ref <= 5e-3
    assert r_ub <= 5e-3


@pytest.mark.parametrize("prec", [Precision.FP64, Precision.FP32, Precision.FP16])
@pytest.mark.parametrize("L", [1, 2, 3, 4])
def test_default_z_chunk_marches_few_planes_twice(prec, L):
    """A chunk of kc planes is marched in kc + 2L-1: on a grid whose tiles
    fill the device several times over, no default chunk is shorter than the
    planes it marches besides its own."""
    g = FDTD(Parameters(256, 256, 256), courant_dt(1, 1, 1), prec)
    g.set_time_blocking_strips(L, 1, 2, 8 if prec == Precision.FP64 else 16)
    assert g.get_time_blocking_strips()["kchunk"] >= 2 * (2 * L - 1)
    g.close()


@pytest.mark.parametrize("shape,L,lanes", [
    ((25, 24, 2000), 4, 32),   # one column more than a 32-lane tile stores
    ((23, 25, 2000), 4, 32),   # one row more
    ((47, 47, 1200), 4, 32),
    ((71, 23, 1500), 4, 32),
    ((25, 25, 2000), 4, 64),
    ((57, 8, 300), 4, 64),     # one column more than a 64-lane tile stores
    ((55, 9, 300), 4, 64),
    ((27, 26, 1800), 3, 32),
    ((59, 11, 40), 3, 64),
    ((29, 28, 1800), 2, 32),
    ((61, 13, 40), 2, 64),
    ((31, 30, 1500), 1, 32),
    ((63, 15, 40), 1, 64),
])
def test_fp64_row_widths(shape, L, lanes):
    """FP64 rows that cannot be staged: tiles of 32 or 64 columns, whichever
    needs fewer plane-rounds, around the tiles' edges, with the shorter passes
    that take the steps left over: the same bits as single sweeps."""
    n, dt = int(np.prod(shape)), courant_dt(1, 1, 1, factor=0.5)
    a, b = (FDTD(Parameters(*shape), dt, Precision.FP64) for _ in range(2))
    for c, v in enumerate(random_state(n, 17)):
        for g in (a, b):
            g.upload(c, v)
    for g in (a, b):
        g.set_point_sources([dict(i=shape[0] - 1, j=q % shape[1], k=(7 * q) % shape[2], comp=q % 3,
                                  kind=0, amp=0.2 / dt) for q in range(70)])
        g.set_probes([(0, 0, 0, 0), (shape[0] - 1, shape[1] - 1, shape[2] - 1, 5)], 4 * L + 6)
    a.set_time_blocking_strips(0)
    b.set_time_blocking_strips(L, 1, 2, 8)
    assert b.get_time_blocking()["lanes"] == lanes
    for steps in (2 * L, L + 2, L + 3):
        a.update_fields(steps)
        b.update_fields(steps)
        assert a.checksum() == b.checksum(), steps
        if steps == L + 2:
            for g in (a, b):
                g.rewind_records()
    assert np.array_equal(a.read_probes(), b.read_probes())
    a.close()
    b.close()


def many_sources(shape, dt, m, plane=None):
    rng = np.random.default_rng(m)
    i, j, k = (rng.integers(0, s, m) for s in shape)
    i[:2], j[:2] = shape[0] - 1, shape[1] - 1
    if plane is not None:
        k[:] = plane
    return [dict(i=int(i[q]), j=int(j[q]), k=int(k[q]), comp=q % 3, kind=1, amp=1e-3 / dt, period=9 * dt,
                 t0=4 * dt, sigma=6 * dt) for q in range(m)]


@pytest.mark.parametrize("prec", [Precision.FP64, Precision.FP32, Precision.FP16])
@pytest.mark.parametrize("shape,m,plane", [
    ((72, 70, 74), 200, 73),    # three to four sources in a row of the last plane
    ((72, 70, 74), 1, 0),
    ((72, 70, 74), 64, None),
    ((101, 99, 12), 65, None),  # one more than a wavefront searches at a time
    ((24, 9, 20), 130, 4),      # rows of the grid that come twice in a tile
    ((7, 5, 20), 40, None),
])
def test_many_sources(prec, shape, m, plane):
    """Passes add the sources of a long list as the sweeps do, cell by cell."""
    dt = courant_dt(1, 1, 1, factor=0.5)
    state = random_state(int(np.prod(shape)), 5)
    a, b = (grid(shape, dt, state, prec, many_sources(shape, dt, m, plane)) for _ in range(2))
    a.set_time_blocking_strips(0)
    b.set_time_blocking_strips(4, 1, 2, 8 if prec == Precision.FP64 else 16)
    for steps in (8, 7, 4):
        a.update_fields(steps)
        b.update_fields(steps)
        assert a.checksum() == b.checksum(), steps
    a.close()
    b.close()


def test_many_sources_in_a_plane_cost_passes_no_more_than_sweeps():
    """Wavefronts pass over the sources of other wavefronts' rows (FP64
    72 x 70 x 74, 200 in one plane, 24 steps: sweeps 1.00 ms, passes 0.70, and
    1.63 where every wavefront took every source of its plane)."""
    shape, dt = (72, 70, 74), courant_dt(1, 1, 1, factor=0.5)
    g = FDTD(Parameters(*shape), dt, Precision.FP64)
    g.set_point_sources(many_sources(shape, dt, 200, 37))
    ms = []
    for L in (4, 0):
        g.set_time_blocking_strips(L, 1, 2, 8)
        g.update_fields(24)
        ms.append(min(g.time_update_fields(24)[0] for _ in range(8)))
    assert ms[0] < 1.1 * ms[1], ms
    g.close()


@pytest.mark.parametrize("prec,shape,m,plane,passes", [
    (Precision.FP32, (101, 99, 97), 500, None, 0),  # 386 us by sweeps, 572 by passes
    (Precision.FP64, (72, 70, 74), 200, None, 0),   # 321, 371
    (Precision.FP32, (101, 99, 97), 16, None, 3),   # 330, 282
    (Precision.FP32, (101, 99, 97), 500, 50, 3),    # 2.52 ms, 1.93
    (Precision.FP64, (101, 99, 97), 200, None, 3),  # 660 us, 570
])
def test_narrow_grids_with_sources_all_over(prec, shape, m, plane, passes):
    """Grids that take passes by default only because these cost less take
    sweeps where sources all over the grid hold the passes up; a blocking that
    was asked for stays."""
    dt = courant_dt(1, 1, 1, factor=0.5)
    state = random_state(int(np.prod(shape)), 5)
    a, b, c = (grid(shape, dt, state, prec, many_sources(shape, dt, m, plane)) for _ in range(3))
    a.set_time_blocking_strips(0)
    c.set_time_blocking_strips(4, 1, 2, 8 if prec == Precision.FP64 else 16)
    for steps in (8, 1, 4):
        for g in (a, b, c):
            g.update_fields(steps)
        assert a.checksum() == b.checksum() == c.checksum(), steps
    assert b.launch_stats()["passes"] == passes
    assert c.launch_stats()["passes"] == 3
    for g in (b, c):  # without its sources a grid is back to passes
        g.set_point_sources([])
        g.update_fields(4)
    assert b.launch_stats()["passes"] == passes + 1
    assert b.checksum() == c.checksum()
    for g in (a, b, c):
        g.close()
