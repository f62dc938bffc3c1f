"""Sizes, values and sequences of calls that went wrong once, in the forms that show it."""
import numpy as np
import pytest

from tests.cases import LX, LZ

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
