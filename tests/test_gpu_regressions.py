"""Sizes, values and sequences of calls that went wrong once, in the forms that show it."""
import threading

import numpy as np
import pytest

from tests.cases import LX, LZ, box, crowded_case, thermal_case

pytestmark = pytest.mark.gpu


def _crowd(shape, cells, seed):
    """Parcels in the given cells only, {(i, j, k): count}, with random values in [0.5, 1]."""
    rng = np.random.default_rng(seed)
    d = np.array([LX / shape[0], LX / shape[1], LZ / shape[2]])
    at = np.concatenate([(np.array(c) + rng.uniform(0.02, 0.98, (m, 3))) * d
                         for c, m in cells.items()])
    n = len(at)
    ic = {k: at[:, a].copy() for a, k in enumerate("xyz")}
    ic["vol"] = rng.uniform(0.5, 1.0, n) * np.prod(d) / 8
    ic.update({k: rng.uniform(0.5, 1.0, n) for k in ("b", "h", "p", "q", "r")})
    return ic, d


def test_crowded_cells_past_2_25():
    """Grids of more than 2^25 cells keep a slot table of 16 entries a cell: cells with more parcels
    than that, below and above the 2^25th.  A node of such a cell is the weighted mean of its 40
    parcels at most: 40 roundings of 6e-8 in each of two sums and the offsets' own (three of 6e-8 a
    weight), of values up to 1, stay below 1e-5."""
    from pmpic_amd.lib import Context
    shape = (512, 512, 129)
    cells = {(5, 7, 3): 40, (100, 200, 128): 40, (300, 17, 128): 17, (511, 511, 128): 33,
             (64, 64, 128): 16}
    assert (128 * 512 + 17) * 512 + 300 >= 1 << 25
    ic, d = _crowd(shape, cells, 11)
    g = Context(*shape, 0.0, LX, 0.0, LX, 0.0, LZ, 4096, precision=1)
    g.set_parcels(ic)
    for _ in range(2):  # the second call finds what the first left behind
        g.writebinary_grids()
    first = 0
    grids = {k: g.grid(k) for k in ("p", "hg")}
    g.close()
    for c, m in cells.items():
        s = slice(first, first + m)
        first += m
        f = [ic[k][s] / d[a] - c[a] for a, k in enumerate("xyz")]
        for bits in range(8):
            b = [(bits >> a) & 1 for a in range(3)]
            w = ic["vol"][s] * np.prod([f[a] if b[a] else 1 - f[a] for a in range(3)], axis=0)
            i, j = (c[0] + b[0]) % 512 + 2, (c[1] + b[1]) % 512 + 2
            for name, field in (("p", "p"), ("hg", "h")):
                want = np.sum(w * ic[field][s]) / np.sum(w)
                assert abs(grids[name][i, j, c[2] + b[2]] - want) < 1e-5, (c, bits, name)


@pytest.mark.parametrize("slots", ["16", "32"])
@pytest.mark.parametrize("nx", [18, 32])
@pytest.mark.parametrize("where", ["between_steps", "stage_1", "stage_3"])
def test_set_time_between_components(monkeypatch, nx, slots, where):
    """pmpic_set_time with the values that stand already changes nothing, wherever a caller puts it:
    after a vort2vel that has used up the lists of crowded cells, between steps (with a grid export,
    which waits for the device) or between the components of a stage.  The runs stay bit-identical."""
    from pmpic_amd.lib import Context
    monkeypatch.setenv("PMPIC_SLOT_CAPACITY", slots)
    shape = (nx, 12, 8)
    ic = crowded_case(*shape)
    for k in "pqr":
        ic[k] = 10.0 * ic[k]
    b = box(*shape)
    runs = []
    for _ in range(2):
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    3 * len(ic["x"]), precision=1)
        g.set_parcels(ic)
        runs.append(g)

    def set_same_time(g):
        g.grid("p")
        g.set_time(g.time, g.dtm)

    for s in range(3):
        for i, g in enumerate(runs):
            if where == "between_steps":
                if i:
                    g.vort2vel()
                    set_same_time(g)
                g.step()
                continue
            for stage in (1, 2, 3, 4):
                g.vort2vel()
                if i and where == f"stage_{stage}":
                    set_same_time(g)
                g.vorticity_tendency()
                g.rk4_integrator()
                g.parcel_splitting()
                g.parcel_mixing()
        assert runs[0].n == runs[1].n
        want, got = (g.get_parcels() for g in runs)
        for k in want:
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"step {s}: {k}")
        for k in ("u", "v", "w", "p", "q", "r", "b"):
            np.testing.assert_array_equal(runs[1].grid(k), runs[0].grid(k), err_msg=f"{s}: {k}")
    for g in runs:
        g.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_set_time_sets_the_step(precision):
    """The timestep given between vorticity_tendency, which selects one at stage 1, and
    rk4_integrator is the one that the stage takes."""
    from pmpic_amd.lib import Context
    shape = (12, 10, 8)
    ic = crowded_case(*shape, extra=(3,))
    b = box(*shape)
    g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                3 * len(ic["x"]), precision=precision)
    g.set_parcels(ic)
    g.vort2vel()
    g.vorticity_tendency()
    g.set_time(1.5, 0.00125)
    assert g.state()[1:] == (1.5, 0.00125)
    g.rk4_integrator()
    assert g.state()[1:] == (1.5, 0.00125)
    g.close()


@pytest.mark.parametrize("value", [np.inf, -np.inf, 1e308, -1e308, 1e300])
@pytest.mark.parametrize("axis,status", [("x", 1), ("y", 2), ("z", 3)])
def test_positions_without_a_cell_are_refused(axis, status, value):
    """An infinite position, one whose quotient by the cell size overflows and one that does not:
    refused in every call that finds a parcel's cell, out of the box or (4, above the box by more cells
    than an integer holds) by its offset."""
    from pmpic_amd.lib import Context, PmpicError
    shape = (12, 10, 8)
    ic = crowded_case(*shape, extra=(3,))
    n = len(ic["x"])
    ic[axis] = ic[axis].copy()
    ic[axis][n // 2] = value
    b = box(*shape)
    g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"], 3 * n)
    calls = {"cache_weights": g.cache_weights, "par2grid": lambda: g.par2grid(np.ones(n)),
             "grid2par": lambda: g.grid2par(np.ones(g.gshape)),
             "writebinary_grids": g.writebinary_grids, "step": g.step}
    for name, call in calls.items():
        g.set_parcels(ic)
        with pytest.raises(PmpicError) as e:
            call()
        assert e.value.status in (status, 4 if value == 1e300 else status), name
    g.close()


def _noalloc_pair(shape, ppc, seed):
    """A context, a call of the allocation-free par2grid of its buoyancy (its status and grid) and
    the grid that pmpic_par2grid gives."""
    from pmpic_amd.lib import Context
    from tests.test_zz_no_alloc import _noalloc
    ic = thermal_case(*shape, ppc, seed=seed, vort=1.0)
    b = box(*shape)
    g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                len(ic["x"]) + 64)
    g.set_parcels(ic)
    return g, ic, lambda: _noalloc(g, ic["b"]), g.par2grid(ic["b"])


def test_noalloc_calls_of_two_threads():
    """Allocation-free calls of two contexts, a large and a small one, at the same time, then one
    after another: all bit-identical to pmpic_par2grid."""
    pairs = [_noalloc_pair((32, 32, 32), 3, 21), _noalloc_pair((10, 12, 5), 2, 22)]
    bad = []

    def run(call, want):
        for _ in range(50):
            st, got = call()
            if st != 0 or not np.array_equal(got, want):
                bad.append(st)

    th = [threading.Thread(target=run, args=p[2:]) for p in pairs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for g, _, call, want in pairs:
        st, got = call()
        assert st == 0
        np.testing.assert_array_equal(got, want)
        g.close()


def test_noalloc_after_a_refused_call():
    """A call that fails on a parcel outside the box leaves nothing to the next one."""
    g, ic, call, want = _noalloc_pair((12, 10, 8), 2, 23)
    out_of_box = dict(ic, z=ic["z"].copy())
    out_of_box["z"][7] = 2 * LZ
    g.set_parcels(out_of_box)
    assert call()[0] == 3  # PMPIC_ERR_OUT_OF_BOX_Z
    g.set_parcels(ic)
    st, got = call()
    assert st == 0
    np.testing.assert_array_equal(got, want)
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [32_767, 32_768, 131_071, 131_072, 2_097_151, 2_097_152])
def test_parcel_arrays_around_the_copy_rules(n, precision):
    """Parcel arrays there and back either side of the parts that go through pinned slots to the host
    (256 KB of 17, or 1 MB where each is taken alone, which 16 MB are by four threads):
    equal in the FP64 form, rounded to FP32 in the other (cells of unit size, positions in the first)."""
    from pmpic_amd.lib import PARCEL_FIELDS, Context
    rng = np.random.default_rng(n)
    ic = {k: rng.uniform(0.1, 0.9, n) for k in PARCEL_FIELDS}
    g = Context(8, 6, 5, 0.0, 8.0, 0.0, 6.0, 0.0, 5.0, n, precision=precision)
    for _ in range(2):
        g.set_parcels(ic)
        got = g.get_parcels()
    g.close()
    for k in PARCEL_FIELDS:
        want = ic[k] if precision == 0 or k == "tag" else ic[k].astype(np.float32)
        np.testing.assert_array_equal(got[k], want.astype(np.float64), err_msg=k)


@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("stage", [1, 2, 3, 4])
def test_parcels_that_would_leave_the_box_stay(monkeypatch, stage, fused):
    """An FP32-bulk stage whose timestep takes parcels out of the box (by thousands of cells, where
    they have a vertical velocity to speak of) reports it and leaves those parcels as they were, in
    either of the two sets that the stages write, and in the next par2grid."""
    from pmpic_amd.lib import Context, PmpicError
    monkeypatch.setenv("PMPIC_FUSED_BINNING", fused)
    shape = (12, 10, 8)
    ic = thermal_case(*shape, 2, vort=2.0)
    b = box(*shape)
    g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                3 * len(ic["x"]), precision=1)
    g.set_parcels(ic)
    g.step(2)

    for _ in range(stage - 1):
        g.vort2vel()
        g.vorticity_tendency()
        g.rk4_integrator()
        g.parcel_splitting()
        g.parcel_mixing()
    g.vort2vel()
    g.vorticity_tendency()
    before = g.get_parcels()
    g.set_time(g.time, 1e6)
    with pytest.raises(PmpicError) as e:
        g.rk4_integrator()
    assert e.value.status == 3  # PMPIC_ERR_OUT_OF_BOX_Z
    after = g.get_parcels()
    where = ("x", "y", "z", "p", "q", "r")
    stayed = np.all([after[k] == before[k] for k in where], axis=0)
    assert stayed.mean() > 0.9
    # and they are in the lists: a grid of the parcels is that of a context given them as they are
    g.writebinary_grids()
    got = {k: g.grid(k) for k in ("b", "hg", "p", "q", "r")}
    h = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                3 * len(ic["x"]), precision=1)
    h.set_parcels(after)
    h.writebinary_grids()
    for k, want in got.items():
        assert np.abs(h.grid(k) - want).max() <= 1e-5 * max(1.0, np.abs(want).max()), k
    g.close()
    h.close()


@pytest.mark.parametrize("n", [0, 1, 2, 1001, 65_536, 65_537])
@pytest.mark.parametrize("precision", [0, 1])
def test_conservation_sums_in_parcel_order(n, precision):
    """The volume integrals, compensated (Neumaier) in parcel order: bit for bit what the same
    additions give here, of the values as the form holds them, large and small ones mixed."""
    from pmpic_amd.lib import Context
    rng = np.random.default_rng(n)
    ic = {k: rng.uniform(0.1, 0.9, n) for k in "xyz"}
    for k in ("vol", "b", "h", "p", "q", "r"):
        ic[k] = rng.standard_normal(n) * 10.0 ** rng.integers(-6, 7, n)
    g = Context(8, 6, 5, 0.0, 8.0, 0.0, 6.0, 0.0, 5.0, n + 1, precision=precision)
    g.set_parcels(ic)
    held = g.get_parcels()
    got = g.conservation_sums()
    g.close()
    for k, name in enumerate((None, "b", "h", "p", "q", "r")):
        s = comp = 0.0
        for v, f in zip(held["vol"], held[name] if name else np.ones(n)):
            term = float(v * f)
            t = s + term
            comp += (s - t) + term if abs(s) >= abs(term) else (term - t) + s
            s = t
        assert got[k] == s + comp, name


@pytest.mark.parametrize("nz", [63, 64])
def test_absorption_from_either_kind_of_list(monkeypatch, nz):
    """Mixing either side of 2^17 tiles, where the absorption looks at one or at eight of them a
    wavefront, with a slot table and without one: the lists are laid out and found in other ways, but
    each parcel absorbs once, so the parcels stay bit-identical."""
    from pmpic_amd.lib import Context
    shape = (128, 128, nz)
    ic = thermal_case(*shape, 2, vort=1.0, shrink=0.02, thin=0.02, near_split=0.01)
    b = box(*shape)
    want = None
    for slots in ("0", "16"):
        monkeypatch.setenv("PMPIC_SLOT_CAPACITY", slots)
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    2 * len(ic["x"]), precision=1)
        g.set_parcels(ic)
        changed = 0
        for _ in range(2):
            g.step()
            changed += sum(g.last_counts()[1:])
        assert changed > 0
        got = g.get_parcels(["x", "z", "p", "q", "r", "b", "h", "vol", "tag"])
        g.close()
        if want is None:
            want = got
            continue
        for k in want:
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("nz", [63, 64])
def test_absorption_against_fp64(nz):
    """The mixing alone, of the same parcels, in both forms, either side of 2^17 tiles: the same
    parcels removed and added, and the kept ones' volumes within 5e-6 (a volume and eight shares of at
    most 1e-2 of it, each within some 64 roundings of 6e-8; a share taken twice or left out is a few
    1e-4)."""
    from pmpic_amd.lib import Context
    shape = (128, 128, nz)
    ic = thermal_case(*shape, 2, vort=1.0, shrink=0.02, thin=0.02)
    b = box(*shape)
    out = []
    for precision in (0, 1):
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    2 * len(ic["x"]), precision=precision)
        g.set_parcels(ic)
        for _ in range(4):  # the component acts in every fourth call
            g.parcel_mixing()
        out.append((g.n, g.last_counts(), g.get_parcels(["vol", "tag"])))
        g.close()
    assert out[0][:2] == out[1][:2] and min(out[0][1][1:]) > 0
    vol64, vol32 = out[0][2]["vol"], out[1][2]["vol"]
    assert np.array_equal(out[0][2]["tag"], out[1][2]["tag"])
    assert np.abs(vol32 / vol64 - 1).max() < 5e-6
    change = np.abs(vol64 / ic["vol"].max() - 1)
    assert change[change < 0.05].max() > 1e-4  # something was absorbed


@pytest.mark.parametrize("precision", [0, 1])
def test_grids_of_a_new_context_are_zero(precision):
    """Grids exported, and tendencies taken, before the first vort2vel: zero, not what the memory held
    for a context before (whose grids are far from it)."""
    from pmpic_amd.lib import GRID_IDS, Context
    shape = (32, 24, 16)
    b = box(*shape)
    ic = thermal_case(*shape, 2, vort=3.0)
    for fresh in (False, True):
        g = Context(*shape, b["xmin"], b["xmax"], b["ymin"], b["ymax"], b["zmin"], b["zmax"],
                    2 * len(ic["x"]), precision=precision)
        if not fresh:
            g.set_parcels(ic)
            g.step()
        else:
            for _ in range(2):
                for k in GRID_IDS:
                    assert not g.grid(k).any(), k
                g.vorticity_tendency()
            assert g.dtm == 0.01
        g.close()
