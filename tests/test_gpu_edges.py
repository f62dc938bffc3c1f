"""The kernels at the edges of their tiles, chunks and dispatch rules, against the oracle.

par2grid: x rows shorter, equal and longer than the eight-cell tiles; cells of 0, 1, 7, 8, 9, 63,
64, 65 and 130 parcels (chunks of eight, ordered lists of up to 64 in LDS, longer in memory), with
the parcels in and out of slot order, and parcel counts either side of the binning walks' rule.
The bar is 1e-12 of the field's maximum, as for every FP64 par2grid; each cell holds few enough
parcels that sums of 1e3 terms with 1e-16 rounding stay far below it.

The column kernel: levels per column below, at and above its read-ahead (8), rows of wavenumber
blocks below and above a wavefront's 16, whole steps, 1e-12 (FP64) and 1e-5 (FP32-bulk against
FP64, that form's bar).

The FP32-bulk accumulation: the same tiles and occupancies, and those around its slot capacities.

The haloswap's permutation: parcel counts either side of a block, of the staging that needs no
count read back (2^20 parcels) and of the one-launch scan (16,384 blocks).
"""
import numpy as np
import pytest

from tests.cases import box, rel_err, thermal_case

pytestmark = pytest.mark.gpu

OCCUPANCY = (0, 1, 7, 8, 9, 63, 64, 65, 130)


def _pair(oracle_mod, shape, ic, precision=0):
    from pmpic_amd.lib import Context
    b = box(*shape)
    args = (*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
            2 * len(ic["x"]) + 64)
    o = oracle_mod.Oracle(*args, 0.01, 0.01, 0.5)
    g = Context(*args, precision=precision)
    o.set_parcels(ic)
    g.set_parcels(ic)
    return o, g


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("nx", [2, 3, 8, 9, 10, 15, 16, 18, 25])
def test_par2grid_tiles_and_occupancy(oracle_mod, nx, shuffled, bar):
    shape = (nx, 4, 3)
    b = box(*shape)
    rng = np.random.default_rng(nx)
    d = [(b[k + "max"] - b[k + "min"]) / n for k, n in zip("xyz", shape)]
    at = []
    for c in range(nx * 4 * 3):
        m = OCCUPANCY[c % len(OCCUPANCY)]
        ijk = np.array([c % nx, c // nx % 4, c // (nx * 4)])
        at.append((ijk + rng.uniform(0.01, 0.99, (m, 3))) * d)
    at = np.concatenate(at)
    n = len(at)
    if shuffled:
        at = at[rng.permutation(n)]
    ic = dict(x=at[:, 0].copy(), y=at[:, 1].copy(), z=at[:, 2].copy(),
              vol=rng.uniform(0.5, 1.0, n) * np.prod(d) / 8)
    o, g = _pair(oracle_mod, shape, ic)
    o.cache_weights()
    for _ in range(2):  # the second call finds what the first left behind
        var = rng.standard_normal(n)
        bar("par2grid", rel_err(g.par2grid(var)[2:-2, 2:-2], o.par2grid(var)[2:-2, 2:-2]), 1e-12)
    g.close()


@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("most", [1 << 19, 1 << 22])
def test_par2grid_binning_walks(oracle_mod, most, extra, bar):
    """Parcel counts at the changes of the binning's walk length."""
    shape = (32, 32, 32)
    rng = np.random.default_rng(1)
    b = box(*shape)
    n = most + extra
    ic = {k: rng.uniform(b[k + "min"], b[k + "max"] * (1 - 1e-9), n) for k in "xyz"}
    ic["vol"] = np.full(n, 1e-3)
    o, g = _pair(oracle_mod, shape, ic)
    o.cache_weights()
    var = np.cos(ic["x"]) * ic["z"]
    bar("par2grid", rel_err(g.par2grid(var)[2:-2, 2:-2], o.par2grid(var)[2:-2, 2:-2]), 1e-12)
    g.close()


@pytest.mark.parametrize("shape", [(8, 8, 2), (8, 9, 3), (15, 8, 7), (16, 10, 8), (30, 6, 9),
                                   (32, 8, 15), (36, 5, 16), (64, 4, 17)])
def test_column_kernel_lengths(oracle_mod, shape, bar):
    ic = thermal_case(*shape, 2, vort=1.0)
    o, g = _pair(oracle_mod, shape, ic)
    _, f = _pair(oracle_mod, shape, ic, precision=1)
    for _ in range(2):
        o.step()
        g.step()
        f.step()
    for k in ("u", "v", "w", "p", "q", "r"):
        want = o.grid(k)[2:-2, 2:-2]
        bar(k, rel_err(g.grid(k)[2:-2, 2:-2], want), 1e-12)
        bar(k + "32", rel_err(f.grid(k)[2:-2, 2:-2], want), 1e-5)
    for k in ("u_s", "v_s", "w_s"):
        bar(k, rel_err(g.spectral(k), o.spec(k)), 1e-12)
    g.close()
    f.close()


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4096, 1_048_576, 1_048_577, 4_194_304, 4_194_305])
@pytest.mark.parametrize("crossing", [0.0, 0.003, 0.5])
def test_haloswap_counts(n, crossing):
    """The haloswap's permutation either side of its scan's and its staging's rules: crossing
    parcels, shifted by a period, in (direction, slot) order in the vacated slots.  Tags are whole
    numbers; a position takes two additions of up to two periods, so it comes back to within 8
    roundings of a period."""
    from pmpic_amd.lib import Context
    b = box(8, 6, 5)
    lx, ly = b["xmax"] - b["xmin"], b["ymax"] - b["ymin"]
    rng = np.random.default_rng(n)
    ic = dict(x=b["xmin"] + rng.uniform(0.01, 0.99, n) * lx,
              y=b["ymin"] + rng.uniform(0.01, 0.99, n) * ly,
              z=b["zmin"] + rng.uniform(0.1, 0.9, n) * (b["zmax"] - b["zmin"]),
              tag=np.arange(n, dtype=np.float64))
    step = [rng.choice([-1, 0, 1], n, p=[crossing / 2, 1 - crossing, crossing / 2])
            for _ in range(2)]
    x = ic["x"] + step[0] * lx
    y = ic["y"] + step[1] * ly
    # N, NE, E, SE, S, SW, W, NW
    order = {(0, 1): 1, (1, 1): 2, (1, 0): 3, (1, -1): 4, (0, -1): 5, (-1, -1): 6, (-1, 0): 7,
             (-1, 1): 8, (0, 0): 0}
    table = np.array([[order[(i, j)] for j in (-1, 0, 1)] for i in (-1, 0, 1)])
    direction = table[step[0] + 1, step[1] + 1]
    slots = np.flatnonzero(direction)
    moved = slots[np.argsort(direction[slots], kind="stable")]
    tag = ic["tag"].copy()
    tag[slots] = ic["tag"][moved]
    g = Context(8, 6, 5, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"], n + 64)
    g.set_parcels(dict(ic, x=x, y=y))
    g.parcel_haloswap()
    out = g.get_parcels()
    assert np.array_equal(out["tag"], tag)
    back = np.argsort(tag)
    for k, start, period in (("x", ic["x"], lx), ("y", ic["y"], ly)):
        assert np.abs(out[k][back] - start).max() <= 8 * np.finfo(float).eps * period
    g.close()


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("slots", ["16", "32", "0"])
@pytest.mark.parametrize("nx", [2, 3, 8, 9, 16, 25])
def test_bulk32_tiles_and_occupancy(monkeypatch, nx, slots, shuffled):
    """The FP32-bulk accumulation and its lists (slot table, overflow region, LDS and memory
    orderings) against the FP64 form.  A node adds up to 8 cells of up to 300 parcels: a chain of
    300 roundings of 6e-8 is 1.8e-5 of values between 0.5 and 1, so 3.6e-5 of a grid's least
    maximum."""
    from pmpic_amd.lib import Context
    monkeypatch.setenv("PMPIC_SLOT_CAPACITY", slots)
    occupancy = (0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 300)
    shape = (nx, 4, 3)
    b = box(*shape)
    rng = np.random.default_rng(nx)
    d = [(b[k + "max"] - b[k + "min"]) / n for k, n in zip("xyz", shape)]
    at = []
    for c in range(nx * 4 * 3):
        ijk = np.array([c % nx, c // nx % 4, c // (nx * 4)])
        at.append((ijk + rng.uniform(0.01, 0.99, (occupancy[c % len(occupancy)], 3))) * d)
    at = np.concatenate(at)
    n = len(at)
    if shuffled:
        at = at[rng.permutation(n)]
    ic = dict(x=at[:, 0].copy(), y=at[:, 1].copy(), z=at[:, 2].copy(),
              vol=rng.uniform(0.5, 1.0, n) * np.prod(d) / 8,
              **{k: rng.uniform(0.5, 1.0, n) for k in ("b", "h", "p", "q", "r")})
    grids = []
    for precision in (0, 1):
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    2 * n + 64, precision=precision)
        g.set_parcels(ic)
        for _ in range(2):  # the second call finds what the first left behind
            g.writebinary_grids()
        grids.append({k: g.grid(k)[2:-2, 2:-2] for k in ("b", "hg", "p", "q", "r")})
        g.close()
    for k, want in grids[0].items():
        assert rel_err(grids[1][k], want) < 3.6e-5, k


@pytest.mark.parametrize("nx,ny", [(2, 2), (2, 5), (5, 2), (3, 16), (16, 32), (18, 32), (25, 16),
                                   (45, 27), (64, 60), (60, 64), (64, 64), (81, 48)])
def test_plane_transforms(nx, ny):
    """Both transforms at the smallest planes, the change of workgroup (512 points) and the largest
    plane that fits one (60 x 64 in FP64), against numpy: FP64 sums of a few thousand terms, 1e-13
    of the maximum."""
    from pmpic_amd.lib import Context
    b = box(nx, ny, 3)
    g = Context(nx, ny, 3, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"], 64)
    rng = np.random.default_rng(nx * ny)
    field = np.zeros(g.gshape)
    field[2:-2, 2:-2] = rng.standard_normal(field[2:-2, 2:-2].shape)
    got = g.fft_forward(field)
    y = np.fft.rfft(field[2:-2, 2:-2], axis=1)  # [x, y, z]
    want = np.zeros_like(got)
    for a, part in enumerate((y.real, y.imag)):
        x = np.fft.rfft(part, axis=0)
        want[0::2, a::2], want[1::2, a::2] = x.real, x.imag
    assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()
    back = g.fft_backward(got)[2:-2, 2:-2]
    assert np.abs(back - field[2:-2, 2:-2]).max() <= 1e-13 * np.abs(field).max()
    g.close()


@pytest.mark.parametrize("shape", [(8, 6, 111), (8, 6, 112), (120, 128, 3), (128, 128, 3)])
def test_column_kernel_split(oracle_mod, shape, bar):
    """Either side of the four-wavefront form's rule: 112 and 113 levels, 248 and 265 tiles."""
    ic = thermal_case(*shape, 1, vort=1.0)
    o, g = _pair(oracle_mod, shape, ic)
    _, f = _pair(oracle_mod, shape, ic, precision=1)
    for c in (o, g, f):
        c.step()
    for k in ("u", "v", "w", "p", "q", "r"):
        want = o.grid(k)[2:-2, 2:-2]
        bar(k, rel_err(g.grid(k)[2:-2, 2:-2], want), 1e-12)
        bar(k + "32", rel_err(f.grid(k)[2:-2, 2:-2], want), 1e-5)
    g.close()
    f.close()


@pytest.mark.parametrize("case,shape", [("8ppc", (32, 16, 8)), ("27ppc", (18, 12, 8)),
                                        ("crowded", (18, 12, 8))])
@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("mixing", [True, False])
def test_moved_entries_change_no_result(monkeypatch, case, shape, fused, mixing):
    """Lists whose entries stages 2 and 4, splitting and mixing move (16 and 32 slots) against lists
    built again each time (no slot table): strong random vorticity and the largest timestep that the
    limits allow, so that many parcels change cell, split and are mixed.  Every list is summed in
    parcel order, so the runs stay bit-identical."""
    from pmpic_amd.lib import Context
    from tests.cases import crowded_case
    ic = (crowded_case(*shape) if case == "crowded" else
          thermal_case(*shape, 3 if case == "27ppc" else 2, vort=30.0, shrink=0.05, thin=0.1,
                       near_split=0.05))
    if case == "crowded":
        for k in "pqr":
            ic[k] = 30.0 * ic[k]
    monkeypatch.setenv("PMPIC_FUSED_BINNING", fused)
    b = box(*shape)
    runs = {}
    for slots in ("0", "16", "32"):
        monkeypatch.setenv("PMPIC_SLOT_CAPACITY", slots)
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    4 * len(ic["x"]), dtm=1.0, dtmax=1.0, mixing=mixing, precision=1)
        g.set_parcels(ic)
        runs[slots] = g
    for s in range(4):
        for g in runs.values():
            g.step()
        want = runs["0"].get_parcels()
        for slots in ("16", "32"):
            g = runs[slots]
            assert (g.n, g.last_counts()) == (runs["0"].n, runs["0"].last_counts()), (slots, s)
            got = g.get_parcels()
            for k in want:
                np.testing.assert_array_equal(got[k], want[k], err_msg=f"{slots} step {s}: {k}")
            for k in ("u", "v", "w", "p", "q", "r", "b"):
                np.testing.assert_array_equal(g.grid(k), runs["0"].grid(k), err_msg=f"{slots} {s}: {k}")
    for g in runs.values():
        g.close()


@pytest.mark.parametrize("n", [7_709, 7_710, 15_420, 123_361, 123_362, 131_072, 131_073, 400_001])
def test_large_host_copies(n):
    """Parcel arrays to the device and back either side of the sizes from which they go through
    pinned slots (1 MB in 17 arrays) and from which several threads carry them (16 MB), with whole and odd last chunks of 1 MB, from two contexts at a
    time: every value comes back as it went."""
    import threading
    from pmpic_amd.lib import PARCEL_FIELDS, Context
    b = box(8, 6, 5)

    def round_trip(seed, out):
        rng = np.random.default_rng(seed)
        ic = {k: rng.standard_normal(n) for k in PARCEL_FIELDS}
        g = Context(8, 6, 5, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"], n)
        for _ in range(2):
            g.set_parcels(ic)
            got = g.get_parcels()
        g.close()
        out.append(all(np.array_equal(got[k], ic[k]) for k in PARCEL_FIELDS))

    out = []
    th = [threading.Thread(target=round_trip, args=(s, out)) for s in (n, n + 1)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert out == [True, True]


@pytest.mark.parametrize("shape", [(128, 128, 63), (128, 128, 64)])
def test_bulk32_mixing_tiles_a_wavefront(shape):
    """Absorption either side of 2^17 tiles, from which a wavefront looks at eight of them: what
    mixing takes from removed parcels and gives to new ones the absorbing parcels make up for, so the
    volume stays (to 1e-6 after three steps, as in the small form of this test), with parcels removed
    and added in one cell of fifty."""
    from pmpic_amd.lib import Context
    ic = thermal_case(*shape, 2, vort=1.0, shrink=0.02, thin=0.02, near_split=0.01)
    b = box(*shape)
    g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                2 * len(ic["x"]), precision=1)
    g.set_parcels(ic)
    s0 = g.conservation_sums()
    changed = 0
    for _ in range(3):
        g.step()
        changed += sum(g.last_counts()[1:])
    s1 = g.conservation_sums()
    g.close()
    assert changed > 0
    assert abs(s1[0] - s0[0]) <= 1e-6 * s0[0]


@pytest.mark.parametrize("change", ["none", "set_parcels", "haloswap", "par2grid", "grids"])
def test_binning_after_mixing(oracle_mod, change, bar):
    """The binning that a mixing without removed or new parcels leaves for the next par2grid, with
    the parcels as they were or changed meanwhile in each way a caller has: against the oracle,
    1e-12."""
    shape = (12, 10, 8)
    ic = thermal_case(*shape, 2, vort=1.0)
    o, g = _pair(oracle_mod, shape, ic)
    for c in (o, g):
        c.step()
    assert g.last_counts() == o.last_counts() == (0, 0, 0)
    if change == "set_parcels":
        other = thermal_case(*shape, 2, seed=9, vort=1.0)
        for c in (o, g):
            c.set_parcels(other)
    elif change == "haloswap":
        for c in (o, g):
            c.parcel_haloswap()
    elif change == "par2grid":
        o.cache_weights()
        var = np.arange(o.n, dtype=np.float64)
        bar("par2grid", rel_err(g.par2grid(var)[2:-2, 2:-2], o.par2grid(var)[2:-2, 2:-2]), 1e-12)
    elif change == "grids":
        g.writebinary_grids()
    for c in (o, g):
        c.step()
    for k in ("u", "v", "w", "p", "q", "r"):
        bar(k, rel_err(g.grid(k)[2:-2, 2:-2], o.grid(k)[2:-2, 2:-2]), 1e-12)
    got, want = g.get_parcels(), o.get_parcels()
    for k in ("x", "y", "z", "p", "q", "r"):
        bar(k, rel_err(got[k], want[k]), 1e-12)
    g.close()


@pytest.mark.parametrize("shape", [(12, 10, 55), (60, 60, 63), (60, 60, 64)])
def test_exports_around_the_pinned_size(oracle_mod, shape, bar):
    """Arrays handed out through pinned memory (up to 2^18 values with halos: 64 x 64 x 64) and
    through a copy: the transforms and exports one after another, none changing the one before
    it, halos included; 1e-12 of the maximum."""
    o, g = _pair(oracle_mod, shape, thermal_case(*shape, ppc_dir=1, vort=0.5))
    grid = np.random.default_rng(7).standard_normal(o.gshape)
    spec, want = g.fft_forward(grid), o.fft_forward(grid)
    back = g.fft_backward(want)
    g.step(1)
    o.step()
    u, v = g.grid("u"), g.grid("v")
    bar("forward", rel_err(spec, want), 1e-12)
    for name, got, ref in (("back", back, o.fft_backward(want)), ("u", u, o.grid("u")),
                           ("v", v, o.grid("v"))):
        inner = ref[2:-2, 2:-2]
        bar(name, rel_err(got, np.pad(inner, ((2, 2), (2, 2), (0, 0)), mode="wrap")), 1e-12)
