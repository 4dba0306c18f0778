"""GPU parity: the HIP path through the C ABI against the FP64 oracle.

Integer/index work (cell keys, sort order, cell tables, neighbour lists with
the 60 cap) must be bit-exact.  Floating-point stages are compared from the
same state (the oracle reads the GPU's FP32 inputs promoted to double); the
tolerance of each comparison is written next to it, and every measured error
is appended to the error log of gpu_common (ERR_LOG)."""
import ctypes as C

import numpy as np
import pytest

import orc
from gpu_common import Scene, block_scene, d64, oracle_lists, record, rel_err

pytestmark = pytest.mark.gpu

sa = pytest.importorskip("sphpc_amd")
L = orc.oracle()


def _soa(a):
    a = d64(a)
    return [np.ascontiguousarray(a[:, i]) for i in range(3)]


def _increment_err(v_before, v_after_gpu, v_after_64):
    """Error of a velocity increment stored as v + dv in FP32: returns the
    normwise relative error of dv and the bound 1e-5 max|dv| + 2 ulp(max|v|)
    (the FP32 rounding of v + dv alone is up to half an ulp of |v|)."""
    d_gpu = d64(v_after_gpu) - d64(v_before)
    d_64 = d64(v_after_64) - d64(v_before)
    abs_err = float(np.max(np.abs(d_gpu - d_64)))
    bound = 1e-5 * float(np.max(np.abs(d_64))) + \
        2.0 * float(np.spacing(np.float32(np.max(np.abs(d64(v_after_64))))))
    return abs_err, bound, rel_err(d_gpu, d_64)


# ---------------------------------------------------------------------------
# Native sub-boundary: sort and bounds (thrust_c.cu:86-120)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("adaptive", [False, True])
@pytest.mark.parametrize("n,bits,hi", [(0, 8, 1), (1, 8, 200), (4095, 16, 7),
                                       (4097, 23, 2 ** 23), (100_000, 23, 5000),
                                       (1_000_003, 32, 2 ** 32), (5000, 8, 1)])
def test_sort_by_key_bit_exact(n, bits, hi, adaptive):
    """With the key width given, and with it taken from the keys' OR (all
    keys zero in the last case)."""
    rng = np.random.default_rng(n)
    keys = rng.integers(0, min(hi, 2 ** bits), n, dtype=np.uint64).astype(np.uint32)
    vals = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    k, v = sa.sort_by_key(keys, vals, key_bits=None if adaptive else bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k, keys[order])
    assert np.array_equal(v, vals[order])
    if n:
        k2, v2 = keys.copy(), vals.copy()
        L.orc_sort_by_key(n, k2, v2)
        assert np.array_equal(k, k2) and np.array_equal(v, v2)


@pytest.mark.parametrize("bits", [1, 9, 10, 11, 17, 20, 21, 30, 31])
@pytest.mark.parametrize("n", [2, 8 * 4096, 8 * 4096 + 1, 32 * 4096 + 1, (1 << 21) + 1])
def test_sort_at_the_limits_of_its_digits(n, bits):
    """10-bit digits where they save a pass, up to 2^21 pairs; rows of the
    histogram summed by the blocks themselves up to 8 (10 bits) or 32 tiles."""
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(np.uint32)
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    order = np.argsort(keys, kind="stable")
    for kb in (bits, None):
        k, v = sa.sort_by_key(keys, vals, kb)
        assert np.array_equal(k, keys[order]) and np.array_equal(v, vals[order])


@pytest.mark.parametrize("n", [63, 64, 65, 100_001])
def test_cell_bounds_of_unsorted_keys(n):
    """The bounds count, so keys in any order give the same table; runs of equal
    keys across wavefronts and at the ragged end."""
    keys = np.random.default_rng(n).integers(0, 7, n).astype(np.uint32)
    keys[-3:] = 6
    lo, hi = sa.cell_bounds(keys, 6)
    c, k = np.arange(6, dtype=np.uint32), np.sort(keys)
    assert np.array_equal(lo, np.searchsorted(k, c, "left"))
    assert np.array_equal(hi, np.searchsorted(k, c, "right"))


@pytest.mark.parametrize("n,cells", [(0, 10), (1, 1), (5000, 997), (300_000, 1_000_000)])
def test_cell_bounds_bit_exact(n, cells):
    rng = np.random.default_rng(cells)
    keys = np.sort(rng.integers(0, cells + 5, n).astype(np.uint32))  # some keys >= cells
    lo, hi = sa.cell_bounds(keys, cells)
    c = np.arange(cells, dtype=np.uint32)
    assert np.array_equal(lo, np.searchsorted(keys, c, "left"))
    assert np.array_equal(hi, np.searchsorted(keys, c, "right"))


@pytest.mark.parametrize("cells", [4095, 4096, 4097, 8 * 4096, 8 * 4096 + 1, 2048 * 4096,
                                   2048 * 4096 + 1])
def test_cell_bounds_at_the_edges_of_the_scan(cells):
    """The scan's tiles of 4096 cells and its two limits: up to 8 tiles sum the
    input itself, up to 2048 the tiles' sums."""
    test_cell_bounds_bit_exact(20_000, cells)


@pytest.mark.parametrize("cells", [256 * 4096, 256 * 4096 + 1, 257 * 4096 + 2, 700 * 4096 + 3])
def test_cell_bounds_of_mostly_empty_tables(cells):
    """Past 256 tiles of 4096 cells a tile without keys is not read; ends that are
    no multiple of four, keys in a few tiles, the first and the last cell."""
    rng = np.random.default_rng(cells)
    keys = np.concatenate([np.zeros(3), rng.integers(4095, 4098, 50),
                           rng.integers(130 * 4096, 131 * 4096, 5000), np.full(7, cells - 1)])
    keys = np.sort(keys).astype(np.uint32)
    lo, hi = sa.cell_bounds(keys, cells)
    c = np.arange(cells, dtype=np.uint32)
    assert np.array_equal(lo, np.searchsorted(keys, c, "left"))
    assert np.array_equal(hi, np.searchsorted(keys, c, "right"))


@pytest.mark.parametrize("n,cap", [(1, 1), (3, 7), (4, 4), (1021, 2000), ((1 << 17) - 1,) * 2,
                                   (1 << 17,) * 2, (5, 1 << 17), (32769, 1 << 17),
                                   ((1 << 19) + 1,) * 2,
                                   ((1 << 21) + 5,) * 2])
def test_state_transfer_round_trip(n, cap):
    """One chunk below 2^17 particles of capacity, up to 16 above, ragged ends,
    and a download of some of the arrays only."""
    sc = Scene(0.02, (1.0, 1.0, 1.0))
    rng = np.random.default_rng(n)
    pos, vel = rng.random((n, 3), np.float32), rng.standard_normal((n, 3), np.float32)
    with sc.context(cap) as ctx:
        for _ in range(2):
            ctx.upload(pos, vel)
            p, v = ctx.download()
            assert np.array_equal(p, pos) and np.array_equal(v, vel)
            pos, vel = vel, pos
        y, vz = np.full(n, 7.0, np.float32), np.full(n, 7.0, np.float32)
        for some in ((y, None), (y, vz)):
            a = [None, some[0], None, None, None, some[1]]
            sa.check(sa.lib().sph_download_state(
                ctx.handle, *[sa._fptr(v) if v is not None else None for v in a]))
        assert np.array_equal(y, vel[:, 1]) and np.array_equal(vz, pos[:, 2])


@pytest.mark.parametrize("n,cap", [(3 << 15,) * 2, ((3 << 15) + 1,) * 2, (1 << 15, 1 << 20),
                                   (100001, 100003), (30000, 100003), ((1 << 18) - 1,) * 2,
                                   (1 << 18,) * 2])
def test_state_transfer_at_the_limits_of_its_chunks(n, cap):
    """One chunk up to 3 2^15 particles of capacity, three below 2^18, more from there
    on."""
    test_state_transfer_round_trip(n, cap)


# ---------------------------------------------------------------------------
# Neighbour search in the staged pipeline (neighbors.c:68-298)
# ---------------------------------------------------------------------------
def _scene_dam_block(n=(32, 32, 32), spread=1.0, seed=0, **kw):
    s = 0.02
    sc = Scene(s, (2.0, 1.0, 1.0), **kw)
    pos, vel = block_scene(n, s * spread, (0.0, 0.0, 0.0), jitter=0.01, seed=seed,
                           vel_sigma=0.05, swirl=0.5)
    return sc, pos, vel


def _staged_search(sc, pos, vel, wide=False):
    ctx = sc.context(len(pos))
    ctx.set_tuning(wide_lists=wide)
    ctx.upload(pos, vel)
    ctx.apply_gravity()
    ctx.predict_positions()
    ctx.find_all_neighbors()
    return ctx


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("spread,seed", [(1.0, 0), (0.55, 1)])
def test_neighbor_search_bit_exact(spread, seed, wide):
    """Compact (16-bit offsets) and wide (32-bit) list formats alike."""
    sc, pos, vel = _scene_dam_block(spread=spread, seed=seed)
    ctx = _staged_search(sc, pos, vel, wide)
    n = len(pos)
    # x* against the oracle's ApplyGravity + PredictPositions from the same x, v
    x, y, z = _soa(pos)
    vx, vy, vz = _soa(vel)
    L.orc_apply_gravity(n, vz, C.byref(sc.o))
    xs64 = [np.zeros(n) for _ in range(3)]
    L.orc_predict_positions(n, x, y, z, vx, vy, vz, *xs64, C.byref(sc.o))
    xs_gpu = ctx.field(sa.FIELD_POSITION_STAR)
    err = np.max(np.abs(d64(xs_gpu) - np.stack(xs64, 1)))
    record("predict", abs_err=err)
    assert err <= 4 * np.spacing(np.float32(2.0))  # FP32 x + v dt: a few ulp at |x| <= 2

    # keys, order, cell tables and lists from the GPU's own x*
    xs, ys, zs = _soa(xs_gpu)
    ol = oracle_lists(sc.o, xs, ys, zs)
    k, i = ctx.sorted_pairs()
    assert np.array_equal(k, ol["keys"]) and np.array_equal(i, ol["ids"])
    st, en = ctx.cell_bounds()
    assert np.array_equal(st, ol["start"]) and np.array_equal(en, ol["end"])
    ids, cnt = ctx.neighbors()
    assert np.array_equal(cnt, ol["cnt"])
    assert np.array_equal(ctx.neighbor_counts(), cnt)
    mask = np.arange(orc.MAXN)[None, :] < cnt[:, None]
    assert np.array_equal(ids.reshape(n, -1)[mask], ol["nbr"].reshape(n, -1)[mask])
    st_gpu = ctx.stats()
    assert st_gpu.neighbor_overflow == ol["dropped"]
    assert st_gpu.cell_clamps == 0
    if spread < 1.0:
        assert cnt.max() == orc.MAXN and ol["dropped"] > 0


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 10007])
@pytest.mark.parametrize("cells_used", [1, 3, 4000])
def test_counting_sort_of_scattered_ids(n, cells_used):
    """Stable order whatever the order the counts were taken in: ids scattered
    over few and many cells, whole wavefronts and partial ones."""
    s = 0.02
    sc = Scene(s, (1.0, 0.8, 0.6))
    rng = np.random.default_rng(n + cells_used)
    corner = rng.integers(0, 15, (cells_used, 3)) * sc.h
    pos = (corner[rng.integers(0, cells_used, n)] + rng.uniform(0.1, 0.9, (n, 3)) * sc.h)
    pos = pos.astype(np.float32)
    with sc.context(n) as ctx:
        ctx.upload(pos)
        for _ in range(2):  # the second search finds the counts zero again
            ctx.predict_positions()
            ctx.find_all_neighbors()
            xs, ys, zs = _soa(ctx.field(sa.FIELD_POSITION_STAR))
            keys = np.zeros(n, np.uint32)
            L.orc_hash_particles(n, xs, ys, zs, C.byref(sc.o), keys, np.zeros(n, np.uint32))
            order = np.argsort(keys, kind="stable").astype(np.uint32)
            k, i = ctx.sorted_pairs()
            assert np.array_equal(i, order) and np.array_equal(k, keys[order])
            st, en = ctx.cell_bounds()
            c = np.arange(len(st))
            assert np.array_equal(st, np.searchsorted(k, c, "left"))
            assert np.array_equal(en, np.searchsorted(k, c, "right"))


@pytest.mark.parametrize("crowd", [15, 16, 17, 18, 32, 33, 34, 64, 81, 500])
def test_counting_sort_of_crowded_cells(crowd):
    """Cells of one population, ids scattered over them: a particle's place among its
    cell's ids is counted sixteen at a time past 16, and as scalars by wavefronts that
    lie in one cell."""
    sc = Scene(0.02, (1.0, 0.8, 0.6))
    rng = np.random.default_rng(crowd)
    cells = rng.permutation(1000)[:max(3, 5000 // crowd)]
    corner = np.stack([cells % 10, cells // 10 % 10, cells // 100], 1) * sc.h
    pos = np.repeat(corner, crowd, 0) + rng.uniform(0.1, 0.9, (len(cells) * crowd, 3)) * sc.h
    pos = pos[rng.permutation(len(pos))].astype(np.float32)
    n = len(pos)
    with sc.context(n) as ctx:
        ctx.upload(pos)
        ctx.predict_positions()
        ctx.find_all_neighbors()
        xs, ys, zs = _soa(ctx.field(sa.FIELD_POSITION_STAR))
        keys = np.zeros(n, np.uint32)
        L.orc_hash_particles(n, xs, ys, zs, C.byref(sc.o), keys, np.zeros(n, np.uint32))
        assert set(np.unique(keys, return_counts=True)[1]) == {crowd}
        order = np.argsort(keys, kind="stable").astype(np.uint32)
        k, i = ctx.sorted_pairs()
        assert np.array_equal(i, order) and np.array_equal(k, keys[order])


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("dims", [(1, 1, 1), (13, 5, 1), (34, 34, 35), (35, 35, 34),
                                  (58, 58, 58), (59, 59, 59)])
def test_lists_on_both_sides_of_the_build_kernels_limits(dims, wide):
    """One wave per row up to 40,960 particles, one per dz layer up to 196,608,
    one per 64 particles above; compressed, so that rows hold more than 32
    candidates and lists reach the cap, and with a ragged last group."""
    sc, pos, vel = _scene_dam_block(n=dims, spread=0.5, seed=3)
    ctx = _staged_search(sc, pos, vel, wide)
    n = len(pos)
    ol = oracle_lists(sc.o, *_soa(ctx.field(sa.FIELD_POSITION_STAR)))
    ids, cnt = ctx.neighbors()
    assert np.array_equal(cnt, ol["cnt"])
    mask = np.arange(orc.MAXN)[None, :] < cnt[:, None]
    assert np.array_equal(ids.reshape(n, -1)[mask], ol["nbr"].reshape(n, -1)[mask])
    st = ctx.stats()
    assert st.neighbor_overflow == ol["dropped"] and st.neighbor_pairs == cnt.sum()
    if n > 1000:
        assert cnt.max() == orc.MAXN and ol["dropped"] > 0


@pytest.mark.parametrize("jitter", [0.0, 1e-4, 0.3])
@pytest.mark.parametrize("side", [30, 50, 59])
def test_lists_from_16_bit_coordinates(side, jitter):
    """The list build (one kernel for each side) tests 16-bit coordinates that wrap
    every 8 h, and decides the pairs near h exactly: an exact lattice, whose pairs
    lie at h or a rounding beside it, one barely off it, and a loose one, over 15 to
    29 h.  Particles that are not a number have no neighbours and are nobody's."""
    s = 0.02
    sc = Scene(s, (1.6, 1.6, 1.6))
    pos, vel = block_scene((side,) * 3, s, (0.01, 0.01, 0.01), jitter=jitter, seed=9)
    bad = np.array([0, 1, 2, 3481, 17_777, 17_778, 26_000])
    ctx = _staged_search(sc, pos, vel)
    ol = oracle_lists(sc.o, *_soa(ctx.field(sa.FIELD_POSITION_STAR)))
    ids, cnt = ctx.neighbors()
    assert np.array_equal(cnt, ol["cnt"])
    want, n = ol["nbr"].reshape(len(pos), -1), len(pos)
    mask = np.arange(orc.MAXN)[None, :] < cnt[:, None]
    assert np.array_equal(ids.reshape(n, -1)[mask], want[mask])
    pos[bad[:3], 0] = np.nan
    pos[bad[3:5], 1] = -np.float32(np.nan)
    pos[bad[5:]] = np.nan
    ids, cnt = _staged_search(sc, pos, vel).neighbors()
    mask &= ~np.isin(want, bad)
    mask[bad] = False
    assert np.array_equal(cnt, mask.sum(1))
    got = np.arange(orc.MAXN)[None, :] < cnt[:, None]
    assert np.array_equal(ids.reshape(n, -1)[got], want[mask])


def test_cell_tables_at_the_grid_ends_and_a_crowded_cell():
    """Cell tables from the sorted keys' run ends: runs in the first and the
    last cell of the grid, particles clamped onto the box faces from outside,
    one cell holding 300 particles (five times the list cap), and long stretches
    of empty cells between them."""
    s = 0.02
    sc = Scene(s, (1.0, 1.0, 1.0))
    rng = np.random.default_rng(11)
    h = 2 * s
    crowd = 13 * h + rng.uniform(0.1 * h, 0.9 * h, (300, 3))  # inside cell (13, 13, 13)
    low = rng.uniform(0.0, 0.5 * h, (40, 3))
    high = 1.0 - rng.uniform(0.2 * h, 0.5 * h, (40, 3))
    outside = np.concatenate([rng.uniform(-0.5, -0.1, (20, 3)), rng.uniform(1.1, 1.5, (20, 3))])
    pos = np.concatenate([crowd, low, high, outside]).astype(np.float32)
    pos = pos[rng.permutation(len(pos))]
    vel = np.zeros_like(pos)
    ctx = _staged_search(sc, pos, vel)
    xs_gpu = ctx.field(sa.FIELD_POSITION_STAR)
    xs, ys, zs = _soa(xs_gpu)
    ol = oracle_lists(sc.o, xs, ys, zs)
    k, i = ctx.sorted_pairs()
    assert np.array_equal(k, ol["keys"]) and np.array_equal(i, ol["ids"])
    nx, ny, nz = ctx.grid_dims()
    # the origin cell, and the cell holding the clamped far corner of the box
    c = int((1.0 - 1e-4 * h) // h)
    assert k[0] == 0 and k[-1] == c + c * nx + c * nx * ny
    st, en = ctx.cell_bounds()
    assert np.array_equal(st, ol["start"]) and np.array_equal(en, ol["end"])
    assert (en - st).max() == 300
    ids, cnt = ctx.neighbors()
    assert np.array_equal(cnt, ol["cnt"])
    assert cnt.max() == orc.MAXN and ctx.stats().neighbor_overflow == ol["dropped"]


def test_neighbor_search_long_layers_bit_exact():
    """A bar 8400 particles long and 3 cells thick: a dz layer of the middle
    cell row spans more than 2^16 sorted indices, so those wavefronts (and
    those straddling rows) store 32-bit lists while the others stay compact."""
    s = 0.004
    sc = Scene(s, (34.0, 0.05, 0.05))
    pos, vel = block_scene((8400, 6, 6), s, (0.0, 0.0, 0.0), jitter=0.01, seed=5)
    ctx = _staged_search(sc, pos, vel)
    n = len(pos)
    xs, ys, zs = _soa(ctx.field(sa.FIELD_POSITION_STAR))
    ol = oracle_lists(sc.o, xs, ys, zs)
    # precondition: some particle's layer spans more than 2^16 indices
    o = sc.o
    key = ol["keys"].astype(np.int64)
    cz, rem = key // (o.nx * o.ny), key % (o.nx * o.ny)
    cy, cx = rem // o.nx, rem % o.nx
    y0, y1 = np.maximum(cy - 1, 0), np.minimum(cy + 1, o.ny - 1)
    x0, x1 = np.maximum(cx - 1, 0), np.minimum(cx + 1, o.nx - 1)
    row0 = cz * o.nx * o.ny + y0 * o.nx + x0
    row1 = cz * o.nx * o.ny + y1 * o.nx + x1
    span = ol["end"][row1].astype(np.int64) - ol["start"][row0].astype(np.int64)
    assert span.max() > 2 ** 16 and span.min() < 2 ** 16
    ids, cnt = ctx.neighbors()
    assert np.array_equal(cnt, ol["cnt"])
    mask = np.arange(orc.MAXN)[None, :] < cnt[:, None]
    assert np.array_equal(ids.reshape(n, -1)[mask], ol["nbr"].reshape(n, -1)[mask])
    record("long_layers", particles=n, max_span=int(span.max()))


# ---------------------------------------------------------------------------
# Jacobi stages from the same state (particles.c:461-564)
# ---------------------------------------------------------------------------
def _sphere(dim=64, center=(0.3, 0.3, 0.1), R=0.15):
    wmin = tuple(c - 0.25 for c in center)
    wmax = tuple(c + 0.25 for c in center)
    wmin = (wmin[0], wmin[1], max(wmin[2], 0.0))
    wmax = (wmin[0] + 0.5, wmin[1] + 0.5, wmin[2] + 0.5)
    sdf, dx = orc.sphere_sdf((dim, dim, dim), wmin, wmax, center, R)
    return sdf, (dim, dim, dim), dx, wmin, wmax


@pytest.mark.parametrize("vort_model", [0, 1])
def test_jacobi_stages_match_oracle(vort_model):
    """Density, lambda, delta p and the position update from the same state.
    The Jacobi stages do not read the vorticity model; both settings run."""
    sc, pos, vel = _scene_dam_block(n=(24, 24, 20), seed=3, lambda_eps=600.0, k=0.5, c=0.01,
                               vort_eps=0.01, vort_model=vort_model)
    sdf, dims, dx, wmin, wmax = _sphere()
    o_obs = orc.obstacle(sdf, dims, dx, wmin, wmax)
    ctx = _staged_search(sc, pos, vel)
    ctx.set_obstacle(sdf, dims, dx, wmin, wmax)
    n = len(pos)
    ids, cnt = ctx.neighbors()
    nbr = np.ascontiguousarray(ids)
    cnt = np.ascontiguousarray(cnt)
    for it in range(3):
        xs, ys, zs = _soa(ctx.field(sa.FIELD_POSITION_STAR))
        ctx.compute_densities()
        rho_gpu = ctx.field(sa.FIELD_DENSITY)
        rho64 = np.zeros(n)
        L.orc_compute_densities(n, xs, ys, zs, nbr, cnt, C.byref(sc.o), rho64)
        e_rho = float(np.max(np.abs(rho_gpu - rho64) / rho64))
        # tolerance: 1e-5 relative, per particle
        assert e_rho <= 1e-5, e_rho

        ctx.compute_lambda()
        lam_gpu = ctx.field(sa.FIELD_LAMBDA)
        lam64 = np.zeros(n)
        L.orc_compute_lambda(n, xs, ys, zs, rho64, nbr, cnt, C.byref(sc.o), lam64)
        e_lam = rel_err(lam_gpu, lam64)
        # lambda = -max(C, 0)/(...) with C = rho/rho0 - 1 ~ 1e-3 near rest, the
        # difference of two ~0.8-sized sums: the FP32 rounding of the kernel
        # terms (~1e-7 relative each) moves C by ~1e-7 absolute whatever the
        # summation, so lambda is held normwise (max |d lambda| / max |lambda|)
        # to 1e-5.  Per particle, the relative error is recorded for the
        # particles with |lambda| >= 1% of the maximum.
        assert e_lam <= 1e-5, e_lam
        big = np.abs(lam64) >= 1e-2 * np.max(np.abs(lam64))
        pp = np.abs(d64(lam_gpu) - lam64)[big] / np.abs(lam64[big])
        e_lam_pp_max = float(np.max(pp)) if big.any() else 0.0
        e_lam_pp_med = float(np.median(pp)) if big.any() else 0.0
        e_c = float(np.max(np.abs((d64(rho_gpu) - rho64) / sc.o.rest_density)))

        ctx.update_dps(it)
        dp_gpu = ctx.field(sa.FIELD_DP)
        # isolated: oracle delta p from the GPU's own lambda
        d_iso = [np.zeros(n) for _ in range(3)]
        L.orc_update_dps(n, xs, ys, zs, d64(lam_gpu), nbr, cnt, C.byref(sc.o), it, *d_iso)
        e_dp_iso = rel_err(dp_gpu, np.stack(d_iso, 1))
        assert e_dp_iso <= 1e-5, e_dp_iso
        # compound: oracle delta p from the oracle's lambda
        d64_ = [np.zeros(n) for _ in range(3)]
        L.orc_update_dps(n, xs, ys, zs, lam64, nbr, cnt, C.byref(sc.o), it, *d64_)
        e_dp = rel_err(dp_gpu, np.stack(d64_, 1))

        ctx.update_position_stars()
        xs2_gpu = ctx.field(sa.FIELD_POSITION_STAR)
        x2 = [xs.copy(), ys.copy(), zs.copy()]
        dd = d64(dp_gpu)
        L.orc_update_position_stars(n, *x2, *[np.ascontiguousarray(dd[:, a]) for a in range(3)],
                                    C.byref(sc.o), C.byref(o_obs))
        e_x = float(np.max(np.abs(d64(xs2_gpu) - np.stack(x2, 1))))
        moved = np.max(np.abs(np.stack(x2, 1) - np.stack([xs, ys, zs], 1)))
        record("jacobi", vort_model=vort_model, iteration=it, rho_rel=e_rho,
               lambda_normwise=e_lam, lambda_per_particle_max=e_lam_pp_max,
               lambda_per_particle_median=e_lam_pp_med, C_abs=e_c,
               dp_normwise_isolated=e_dp_iso, dp_normwise=e_dp, x_abs=e_x,
               max_displacement=moved)
        # positions: FP32 rounding of x* + dp plus the collision push
        assert e_x <= 8 * np.spacing(np.float32(1.0)) + 1e-5 * moved, e_x


@pytest.mark.parametrize("vort_model", [0, 1])
def test_velocity_passes_match_oracle(vort_model):
    """Velocity update, both surface-tension passes, XSPH, vorticity and
    confinement from the same state, for the reference's vorticity formula
    (model 0) and the density-weighted one the benchmark runs (model 1)."""
    sc, pos, vel = _scene_dam_block(n=(24, 24, 20), seed=4, lambda_eps=600.0, k=0.5, c=0.01,
                               vort_eps=0.01, vorticity=True, vort_model=vort_model)
    ctx = _staged_search(sc, pos, vel)
    n = len(pos)
    ids, cnt = ctx.neighbors()
    nbr, cnt = np.ascontiguousarray(ids), np.ascontiguousarray(cnt)
    for it in range(2):
        ctx.compute_densities()
        ctx.compute_lambda()
        ctx.update_dps(it)
        ctx.update_position_stars()
    xs, ys, zs = _soa(ctx.field(sa.FIELD_POSITION_STAR))
    xo = _soa(ctx.field(sa.FIELD_POSITION_OLD))
    rho = d64(ctx.field(sa.FIELD_DENSITY))

    ctx.update_velocities()
    v1 = ctx.field(sa.FIELD_VELOCITY)
    o1 = [np.zeros(n) for _ in range(3)]
    L.orc_update_velocities(n, xs, ys, zs, *xo, *o1, C.byref(sc.o))
    # (x* - x)/dt in FP32: x* - x is exact for nearby floats, 1 ulp divide
    e_v = rel_err(v1, np.stack(o1, 1))
    assert e_v <= 1e-6, e_v

    ctx.compute_surface_tension()
    col = ctx.field(sa.FIELD_COLOR)
    v2 = ctx.field(sa.FIELD_VELOCITY)
    c64 = [np.zeros(n) for _ in range(3)]
    L.orc_compute_color(n, xs, ys, zs, rho, nbr, cnt, C.byref(sc.o), *c64)
    e_col = rel_err(col, np.stack(c64, 1))
    assert e_col <= 1e-5, e_col
    vv = _soa(v1)
    cg = _soa(col)
    L.orc_apply_surface_force(n, xs, ys, zs, rho, *cg, nbr, cnt, C.byref(sc.o), *vv)
    a_surf, b_surf, e_surf = _increment_err(v1, v2, np.stack(vv, 1))
    assert a_surf <= b_surf, (a_surf, b_surf)

    ctx.apply_viscosity()
    v3 = ctx.field(sa.FIELD_VELOCITY)
    ov = [np.zeros(n) for _ in range(3)]
    L.orc_apply_viscosity(n, xs, ys, zs, rho, *_soa(v2), nbr, cnt, C.byref(sc.o), *ov)
    a_xsph, b_xsph, e_xsph = _increment_err(v2, v3, np.stack(ov, 1))
    assert a_xsph <= b_xsph, (a_xsph, b_xsph)

    ctx.compute_vorticity()
    w = ctx.field(sa.FIELD_VORTICITY)
    w64 = [np.zeros(n) for _ in range(3)]
    L.orc_compute_vorticity(n, xs, ys, zs, rho, *_soa(v3), nbr, cnt, C.byref(sc.o), *w64)
    e_w = rel_err(w, np.stack(w64, 1))
    # omega sums (v_j - v_i) x gradW: FP32 velocity differences, normwise 1e-5
    assert e_w <= 1e-5, e_w

    ctx.apply_vorticity_confinement()
    v4 = ctx.field(sa.FIELD_VELOCITY)
    vc = _soa(v3)
    L.orc_apply_vorticity_confinement(n, xs, ys, zs, *_soa(w), nbr, cnt, C.byref(sc.o), *vc)
    a_conf, b_conf, e_conf = _increment_err(v3, v4, np.stack(vc, 1))
    assert a_conf <= b_conf, (a_conf, b_conf)

    ctx.update_positions()
    xg, vg = ctx.download()
    assert np.array_equal(xg, np.stack([xs, ys, zs], 1).astype(np.float32))
    assert np.array_equal(vg, v4)
    record("velocity_passes", vort_model=vort_model, v_normwise=e_v, color_normwise=e_col,
           surface_dv_normwise=e_surf, xsph_dv_normwise=e_xsph, vorticity_normwise=e_w,
           confinement_dv_normwise=e_conf)


# ---------------------------------------------------------------------------
# Whole substeps
# ---------------------------------------------------------------------------
def _oracle_state(pos, vel, n):
    x, y, z = _soa(pos)
    vx, vy, vz = _soa(vel)
    arrs = dict(x=x, y=y, z=z, vx=vx, vy=vy, vz=vz, xs=np.zeros(n), ys=np.zeros(n),
                zs=np.zeros(n), density=np.zeros(n), lambda_=np.zeros(n),
                nbr=np.zeros(n * orc.MAXN, np.uint32), cnt=np.zeros(n, np.int32))
    return orc.OrcState(**{k: v.ctypes.data for k, v in arrs.items()}), arrs


@pytest.mark.parametrize("vort_model", [0, 1])
@pytest.mark.parametrize("fused", [True, False])
def test_substep_matches_oracle(fused, vort_model):
    sc, pos, vel = _scene_dam_block(n=(24, 24, 20), seed=5, lambda_eps=600.0, k=0.5, c=0.01,
                               vort_eps=0.01, iters=4, vort_model=vort_model)
    sdf, dims, dx, wmin, wmax = _sphere(center=(0.25, 0.25, 0.05))
    o_obs = orc.obstacle(sdf, dims, dx, wmin, wmax)
    n = len(pos)
    ctx = sc.context(n)
    ctx.upload(pos, vel)
    ctx.set_obstacle(sdf, dims, dx, wmin, wmax)
    if fused:
        ctx.step(1)
    else:
        ctx.apply_gravity(); ctx.predict_positions(); ctx.find_all_neighbors()
        for it in range(sc.iters):
            ctx.compute_densities(); ctx.compute_lambda(); ctx.update_dps(it)
            ctx.update_position_stars()
        ctx.update_velocities(); ctx.compute_surface_tension(); ctx.apply_viscosity()
        ctx.compute_vorticity(); ctx.apply_vorticity_confinement(); ctx.update_positions()
    xg, vg = ctx.download()
    st, a = _oracle_state(pos, vel, n)
    L.orc_substep(n, C.byref(st), C.byref(sc.o), C.byref(o_obs), sc.iters, 0.0, None)
    x64 = np.stack([a["x"], a["y"], a["z"]], 1)
    v64 = np.stack([a["vx"], a["vy"], a["vz"]], 1)
    e_x = float(np.max(np.abs(d64(xg) - x64)))
    e_v = rel_err(vg, v64)
    record("substep_fused" if fused else "substep_staged", vort_model=vort_model, x_abs=e_x,
           v_normwise=e_v)
    # x: a few FP32 ulp at |x| <= 1 plus compounded stage errors
    assert e_x <= 2e-6, e_x
    # v = (x* - x)/dt amplifies the FP32 rounding of x* by 1/dt = 300
    assert e_v <= 2e-4, e_v


def test_fused_equals_staged_closely():
    # vorticity model 1: the reference formula drives |v| to ~1e3 m/s at this
    # scale in one substep, which only magnifies FP32 ordering differences
    sc, pos, vel = _scene_dam_block(n=(20, 20, 16), seed=6, lambda_eps=600.0, k=0.5, c=0.01,
                               vort_eps=0.01, iters=3, vort_model=1)
    n = len(pos)
    out = []
    for fused in (True, False):
        ctx = sc.context(n)
        ctx.upload(pos, vel)
        if fused:
            ctx.step(1)
        else:
            ctx.apply_gravity(); ctx.predict_positions(); ctx.find_all_neighbors()
            for it in range(sc.iters):
                ctx.compute_densities(); ctx.compute_lambda(); ctx.update_dps(it)
                ctx.update_position_stars()
            ctx.update_velocities(); ctx.compute_surface_tension(); ctx.apply_viscosity()
            ctx.compute_vorticity(); ctx.apply_vorticity_confinement(); ctx.update_positions()
        out.append(ctx.download())
    assert np.max(np.abs(out[0][0] - out[1][0])) <= 4 * np.spacing(np.float32(1.0))
    assert rel_err(out[0][1], out[1][1]) <= 1e-4


def test_tolerance_mode_iterations():
    # Plain Jacobi until max density error <= 0.1% (cap 10), the warm-start workload's rule
    sc, pos, vel = _scene_dam_block(n=(24, 24, 24), seed=7, lambda_eps=600.0, iters=10, tol=1e-3)
    n = len(pos)
    ctx = sc.context(n)
    ctx.upload(pos, vel)
    gpu_iters, gpu_err = [], []
    for _ in range(3):
        ctx.step(1)
        s = ctx.stats()
        gpu_iters.append(s.iterations)
        gpu_err.append(s.max_density_error)
        assert s.iterations <= 10
        if s.converged:
            assert s.max_density_error <= 1e-3
    st, a = _oracle_state(pos, vel, n)
    o_iters = []
    for _ in range(3):
        err = C.c_double()
        o_iters.append(L.orc_substep(n, C.byref(st), C.byref(sc.o), None, 10, 1e-3,
                                     C.byref(err)))
    record("tolerance_mode", gpu_iters_0=gpu_iters[0], oracle_iters_0=o_iters[0],
           gpu_iters_2=gpu_iters[2], oracle_iters_2=o_iters[2])
    # iteration counts agree up to one (the 0.1% test of a borderline particle
    # can flip between FP32 and FP64)
    assert all(abs(g - o) <= 1 for g, o in zip(gpu_iters, o_iters)), (gpu_iters, o_iters)


def test_edge_cases_empty_and_single():
    sc = Scene(0.02, (1.0, 1.0, 1.0), iters=3)
    ctx = sc.context(4)
    ctx.upload(np.zeros((0, 3), np.float32))
    ctx.step(2)
    x, v = ctx.download()
    assert x.shape == (0, 3)
    ctx.upload(np.array([[0.5, 0.5, 0.9]], np.float32))
    dt, g = sc.o.dt, sc.o.g
    for step in range(1, 31):
        ctx.step(1)
        x, v = ctx.download()
        expected = 0.9 - g * dt * dt * step * (step + 1) / 2.0
        assert abs(x[0, 2] - expected) < 1e-5
    with pytest.raises(sa.SphError):
        ctx.upload(np.zeros((5, 3), np.float32))


def test_collision_entry_point_matches_oracle():
    dim = (48, 40, 56)
    wmin, wmax = (0.1, 0.2, 0.0), (0.7, 0.7, 0.7)
    center, R = (0.4, 0.45, 0.35), 0.2
    sdf, dx = orc.sphere_sdf(dim, wmin, wmax, center, R)
    rng = np.random.default_rng(11)
    pts = rng.uniform((0.05, 0.15, -0.02), (0.75, 0.75, 0.72), size=(50_000, 3)).astype(np.float32)
    out = sa.collide(pts, sdf, dim, dx, wmin, wmax)
    xs, ys, zs = _soa(pts)
    o = orc.obstacle(sdf, dim, dx, wmin, wmax)
    L.orc_collide(len(pts), xs, ys, zs, C.byref(o))
    ref = np.stack([xs, ys, zs], 1)
    e = float(np.max(np.abs(d64(out) - ref)))
    pushed = np.any(ref != d64(pts), axis=1)
    record("collision", abs_err=e, pushed=int(pushed.sum()))
    assert pushed.sum() > 1000
    # The push is |d| * n with n from central differences of FP32 samples:
    # relative error ~1e-6 of the push distance, plus the FP32 rounding of x.
    push = float(np.max(np.linalg.norm(ref - d64(pts), axis=1)))
    assert e <= 1e-5 * push + 4 * np.spacing(np.float32(1.0)), (e, push)


def test_collision_f64_entry_point_matches_oracle():
    """The FP64-array entry point (the reference's CalculateParticleCollisions
    signature, obstacle_cuda.h:25-29) against the oracle's restatement of the
    reference kernel on the same double arrays: positions outside the
    obstacle's box, or inside it but outside the obstacle, are returned
    bit-for-bit; pushed ones within 1e-5 of the push (FP32 SDF arithmetic)."""
    dim = (48, 40, 56)
    wmin, wmax = (0.1, 0.2, 0.0), (0.7, 0.7, 0.7)
    center, R = (0.4, 0.45, 0.35), 0.2
    sdf, dx = orc.sphere_sdf(dim, wmin, wmax, center, R)
    rng = np.random.default_rng(12)
    pts = rng.uniform((0.05, 0.15, -0.02), (0.75, 0.75, 0.72), size=(50_000, 3))
    # positions FP32 cannot hold: the double coordinates must survive untouched
    pts = pts + 1e-12 * rng.standard_normal(pts.shape)
    out = sa.collide(pts, sdf, dim, dx, wmin, wmax)
    assert out.dtype == np.float64
    xs, ys, zs = [np.ascontiguousarray(pts[:, i]) for i in range(3)]
    o = orc.obstacle(sdf, dim, dx, wmin, wmax)
    L.orc_collide(len(pts), xs, ys, zs, C.byref(o))
    ref = np.stack([xs, ys, zs], 1)
    pushed = np.any(ref != pts, axis=1)
    assert pushed.sum() > 1000
    assert np.array_equal(out[~pushed], pts[~pushed])
    e = float(np.max(np.abs(out - ref)))
    push = float(np.max(np.linalg.norm(ref - pts, axis=1)))
    record("collision_f64", abs_err=e, pushed=int(pushed.sum()),
           bit_identical=float(np.array_equal(out, ref)))
    assert e <= 1e-5 * push, (e, push)


def test_stage_reuse_matches_separate_passes():
    """sph_compute_lambda right after sph_compute_densities takes the lambda
    that the density gather computed, and sph_update_position_stars right after
    sph_update_dps takes the positions that the delta-p pass already updated;
    with a call in between (here downloads) each runs its own pass.  Both give
    the same bits, over two Jacobi iterations with the obstacle, and x* changes
    only at the position stage."""
    sc, pos, vel = _scene_dam_block(n=(24, 24, 20), seed=3, lambda_eps=600.0)
    runs = []
    for interpose in (False, True):
        ctx = _staged_search(sc, pos, vel)
        ctx.set_obstacle(*_sphere())
        out = []
        for it in range(2):
            ctx.compute_densities()
            if interpose:
                ctx.field(sa.FIELD_DENSITY)
            ctx.compute_lambda()
            out.append(ctx.field(sa.FIELD_LAMBDA))
            if interpose:
                x0 = ctx.field(sa.FIELD_POSITION_STAR)
            ctx.update_dps(it)
            if interpose:
                assert np.array_equal(ctx.field(sa.FIELD_POSITION_STAR), x0)
                out.append(ctx.field(sa.FIELD_DP))
            ctx.update_position_stars()
            out.append(ctx.field(sa.FIELD_POSITION_STAR))
        runs.append(out)
        ctx.close()
    # the first run has no delta-p downloads: compare lambda and x* only
    plain = runs[0]
    checked = [a for k, a in enumerate(runs[1]) if k % 3 != 1]
    assert len(plain) == len(checked)
    for a, b in zip(plain, checked):
        assert np.array_equal(a, b)
