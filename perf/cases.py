"""The workloads whose speed is tracked, each through the public entry points of pmpic_amd.

A case is a moist thermal under way in the 2 pi x 2 pi x pi box: parcels on a jittered n x n x n
lattice per cell, a buoyant moist bubble under a stratified layer, and a smooth vorticity field
with a little noise, drawn from a seed.  `stir` cells of smooth displacement plus `stir` / 8
cells of scatter carry the parcels away from the cells they were created in, as in a run that
has been mixing for a while (slot order then no longer follows cell order, the cells are unevenly
filled, and a tenth of the parcels have been split once).

Kinds of case:
  step        a run: `steps` timesteps between two looks at the velocity
  components  the same through the component callbacks one by one, as the Fortran model core
              calls them
  ensemble    `members` thermals on uneven grids stepped together
  restart     parcels uploaded from host arrays, `steps` timesteps with parcels that split, parcels
              below the mixing threshold and thinned cells, every parcel field read back
  dump        the grids of a dump: recomputed from the parcels and read back
  operators   parcel_interpolation_mod and the semi-spectral operators on host arrays
  noalloc     par2grid between device arrays without allocation

Grids and parcels of the FP64 form are returned as they come.  The FP32-bulk form computes in
FP32 and widens on export, so its grids are kept as FP32, and its parcel count (which a
rounding can change by a threshold decision) is left out.
"""
import ctypes
import math

import numpy as np
import torch

from pmpic_amd import lib
from pmpic_amd.config import fortran_real
from pmpic_amd.lib import Context

LX = fortran_real("6.28318531")
LZ = fortran_real("3.14159265")
VELOCITY = ("u", "v", "w")
DUMP = ("u", "v", "w", "p", "q", "r", "b", "hg", "hgliq", "vol")
FP64, FP32 = 0, 1


def listed():
    return [
        # the smallest whole run: a unit-test sized grid, where launches and latency are all
        dict(name="step fp64 12x10x8", kind="step", nx=12, ny=10, nz=8, ppc=2, precision=FP64,
             steps=10, dt=0.001, stir=0.0),
        # the reference's own CPU configuration
        dict(name="step fp64 32^3 27ppc", kind="step", nx=32, ny=32, nz=32, ppc=3, precision=FP64,
             steps=10, dt=0.001, stir=0.0),
        # one small ensemble member run by itself
        dict(name="step fp32 48^3", kind="step", nx=48, ny=48, nz=48, ppc=2, precision=FP32,
             steps=10, dt=0.001, stir=0.0),
        # uneven lengths (x rows not a multiple of a tile, radix 3 and 5), parcels well mixed
        dict(name="step fp32 90x60x41 stirred", kind="step", nx=90, ny=60, nz=41, ppc=2,
             precision=FP32, steps=10, dt=0.001, stir=3.0),
        # eight members of the batched ensemble
        dict(name="ensemble fp32 8 members", kind="ensemble", members=8, steps=5, dt=0.002),
        # the FP32-bulk form's headline configuration
        dict(name="step fp32 256x256x128", kind="step", nx=256, ny=256, nz=128, ppc=2,
             precision=FP32, steps=16, dt=0.01, stir=0.0),
        # the FP64 form's GPU configuration
        dict(name="step fp64 128^3 27ppc", kind="step", nx=128, ny=128, nz=128, ppc=3,
             precision=FP64, steps=6, dt=0.01, stir=0.0),
        # the Fortran model core's call sequence on an uneven grid with mixed parcels
        dict(name="components fp64 45x30x25 stirred", kind="components", nx=45, ny=30, nz=25,
             ppc=3, precision=FP64, steps=2, dt=0.001, stir=3.0),
        # a restart that splits, removes and adds parcels, state out and in through the host
        dict(name="restart fp64 60x48x36", kind="restart", nx=60, ny=48, nz=36, ppc=2,
             precision=FP64, steps=4, dt=0.002, stir=0.0),
        # a grid dump of a mid-sized FP32-bulk run
        dict(name="dump fp32 96x96x64", kind="dump", nx=96, ny=96, nz=64, ppc=2, precision=FP32,
             steps=1, dt=0.01, stir=0.0),
        # host-array operators as other components and the checks use them
        dict(name="operators fp64 64x48x64", kind="operators", nx=64, ny=48, nz=64, ppc=2,
             precision=FP64, stir=1.0),
        # par2grid from inside a loop that must not allocate
        dict(name="noalloc fp64 32^3", kind="noalloc", nx=32, ny=32, nz=32, ppc=2,
             precision=FP64, stir=1.0),
    ]


SMOOTH = [n for n in range(8, 257)
          if not [p for p in (7, 11, 13) + tuple(range(17, 257, 2)) if n % p == 0 and
                  all(p % q for q in range(2, p))]]
MOST = 256 * 256 * 128 * 8  # parcels of the largest listed case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(rng, lo, hi):
    n = _log(rng, lo, hi)
    return min(SMOOTH, key=lambda s: abs(s - n))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["components", "restart", "dump", "operators", "noalloc",
                                      "ensemble"])
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(2, 8), steps=rng.randint(2, 5),
                    dt=round(rng.uniform(0.001, 0.002), 6))
    most = MOST if kind == "step" else 4 << 20
    top = 256 if kind == "step" else 96
    while True:
        nx, ny = _smooth(rng, 10, top), _smooth(rng, 10, top)
        nz = _log(rng, 8, 128 if kind == "step" else 72)
        ppc = rng.choice([2, 2, 3])
        precision = rng.choice([FP64, FP32])
        if kind in ("components", "restart", "operators", "noalloc"):
            precision = FP64
        if kind == "dump":
            precision = FP32
        n = nx * ny * nz * ppc ** 3
        if kind == "noalloc" and (nx * ny * nz > lib.PMPIC_NOALLOC_MAX_CELLS or
                                  n > lib.PMPIC_NOALLOC_MAX_PARCELS):
            continue
        if n <= (most if precision == FP32 else most // 2):
            break
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, ppc=ppc, precision=precision,
                stir=rng.choice([0.0, 0.0, round(rng.uniform(0.5, 4.0), 3)]))
    if kind in ("step", "components", "restart", "dump"):
        case["steps"] = {"step": rng.randint(4, 10), "components": rng.randint(1, 3),
                         "restart": rng.randint(1, 4), "dump": 1}[kind]
        case["dt"] = round(rng.uniform(0.0005, 0.001), 6)
    return case


# ---- inputs -------------------------------------------------------------------------------------
def _parcels(nx, ny, nz, ppc, stir, seed, device, radius=0.8, amplitude=1.0):
    """The parcels of a thermal under way: {field: FP64 tensor}, cell after cell, x fastest."""
    gen = torch.Generator(device=device).manual_seed(int(seed))
    f64 = dict(dtype=torch.float64, device=device)
    dx, dy, dz = LX / nx, LX / ny, LZ / nz
    per, total = ppc ** 3, nx * ny * nz * ppc ** 3

    def uniform(lo, hi):
        return torch.rand(total, generator=gen, **f64).mul_(hi - lo).add_(lo)

    m = torch.arange(total, dtype=torch.int64, device=device)
    cell, sub = m // per, m % per
    x = ((cell % nx).double() + ((sub % ppc).double() + 0.5 + uniform(-0.25, 0.25)) / ppc) * dx
    y = ((cell // nx % ny).double() +
         ((sub // ppc % ppc).double() + 0.5 + uniform(-0.25, 0.25)) / ppc) * dy
    z = ((cell // (nx * ny)).double() +
         ((sub // ppc ** 2).double() + 0.5 + uniform(-0.25, 0.25)) / ppc) * dz
    del m, cell, sub
    vol = torch.full((total,), dx * dy * dz / per, **f64)
    phase = [float(v) for v in torch.rand(6, generator=gen, **f64) * 2 * math.pi]
    if stir:
        def scatter(d):
            return torch.randn(total, generator=gen, **f64).mul_(0.125 * stir * d)
        sx = stir * dx * torch.sin(2 * y + phase[0]) * torch.cos(2 * z) + scatter(dx)
        sy = stir * dy * torch.sin(2 * x + phase[1]) * torch.cos(2 * z) + scatter(dy)
        z = z + stir * dz * torch.sin(x + phase[2]) * torch.sin(y) * torch.sin(z) + scatter(dz)
        x, y = torch.remainder(x + sx, LX), torch.remainder(y + sy, LX)
        z = z.abs()
        z = LZ - (LZ - z).abs()
        z = z.clamp_(1e-9, LZ * (1 - 1e-12))
        x, y = x.clamp_(0.0, LX * (1 - 1e-12)), y.clamp_(0.0, LX * (1 - 1e-12))
        vol = torch.where(uniform(0, 1) < 0.1, 0.5 * vol, vol)
    r2 = (x - LX / 2) ** 2 + (y - LX / 2) ** 2 + (z - 1.0) ** 2
    inside, above = r2 < radius * radius, z >= 1.5
    b = torch.where(inside, amplitude * (1 + 0.01 * uniform(-1, 1)),
                    torch.where(above, z - 1.5, torch.zeros_like(z)))
    h = torch.where(inside, math.exp(-radius) * (1 + 0.01 * uniform(-1, 1)),
                    0.9 * torch.exp(-torch.where(above, z, torch.full_like(z, 1.5))))
    out = dict(x=x, y=y, z=z, b=b, h=h, vol=vol)
    out["p"] = 0.8 * torch.sin(y + phase[3]) * torch.cos(z) + uniform(-0.02, 0.02)
    out["q"] = -0.8 * torch.sin(x + phase[4]) * torch.cos(z) + uniform(-0.02, 0.02)
    out["r"] = 0.4 * torch.cos(x + phase[5]) * torch.cos(y) * torch.sin(z) + uniform(-0.02, 0.02)
    return out


def _events(parcels, case, seed):
    """Parcels about to split, parcels below the mixing threshold, and cells thinned to two."""
    rng = np.random.default_rng(int(seed))
    n, per = len(parcels["x"]), case["ppc"] ** 3
    keep = np.ones((n // per, per), dtype=bool)
    keep[rng.choice(n // per, n // per // 50 + 1, replace=False), 2:] = False
    parcels = {k: v[keep.reshape(-1)] for k, v in parcels.items()}
    n = len(parcels["x"])
    vmin = LX / case["nx"] * (LX / case["ny"]) * (LZ / case["nz"]) / 6. / 6. / 6.
    parcels["vol"][rng.random(n) < 0.02] = 0.5 * vmin
    parcels["stretch"] = np.where(rng.random(n) < 0.02, rng.uniform(3.99, 4.0, n), 0.0)
    parcels["tag"] = np.arange(n, dtype=np.float64)
    return parcels


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _context(case, n):
    cap = int((1.5 if n > 30_000_000 or case["kind"] == "restart" else 2.5) * n) + 4096
    dt = case.get("dt", 0.01)
    return Context(case["nx"], case["ny"], case["nz"], 0.0, LX, 0.0, LX, 0.0, LZ, cap, dtm=dt,
                   dtmax=dt, precision=case["precision"])


def _members(case):
    """Member m's grid, lattice, bubble radius and amplitude."""
    out = []
    for m in range(case["members"]):
        n = (32, 48, 64, 96)[m % 4]
        out.append(dict(nx=n, ny=n, nz=n, ppc=2 if m // 4 % 2 == 0 else 3, precision=FP32,
                        kind="step", dt=case["dt"], stir=0.0, radius=0.5 + 0.06 * m, amplitude=0.5 + 0.18 * m))
    return out


def _host(parcels):
    return {k: v.cpu().numpy() for k, v in parcels.items()}


def _of(case, seed, device=None):
    return _parcels(case["nx"], case["ny"], case["nz"], case["ppc"], case["stir"], seed,
                    device or _device(), case.get("radius", 0.8), case.get("amplitude", 1.0))


def prepare(case, seed):
    if case["kind"] == "ensemble":
        ctxs = []
        for m, member in enumerate(_members(case)):
            ic = _host(_of(member, seed * 64 + m))
            ctxs.append(_context(member, len(ic["x"])))
            ctxs[-1].set_parcels(ic)
        return dict(case=case, ctxs=ctxs)
    ic = _host(_of(case, seed))
    if case["kind"] == "restart":
        ic = _events(ic, case, seed)
    ctx = _context(case, len(ic["x"]))
    ctx.set_parcels(ic)
    state = dict(case=case, ctx=ctx)
    if case["kind"] in ("restart", "components"):
        # the host's own parcel arrays, as long as the model's capacity
        state["mirror"] = {k: np.zeros(ctx.max_parcels) for k in lib.PARCEL_FIELDS}
    if case["kind"] == "restart":
        state["parcels"] = {k: ic.get(k, np.zeros(len(ic["x"]))) for k in lib.PARCEL_FIELDS}
    elif case["kind"] == "dump":
        ctx.step(case["steps"])
    elif case["kind"] == "operators":
        state["var"] = ic["b"]
    elif case["kind"] == "noalloc":
        dev = _device()
        state["var"] = torch.from_numpy(ic["b"]).to(dev)
        state["out"] = torch.empty(ctx.gshape, dtype=torch.float64, device=dev)
    return state


# ---- one pass -----------------------------------------------------------------------------------
def _kept(ctx, name):
    """An exported grid as the program keeps it: the form's own precision."""
    g = torch.from_numpy(ctx.grid(name))
    return g.to(torch.float32) if ctx.precision == FP32 else g


def _look(ctx):
    out = {k: _kept(ctx, k) for k in VELOCITY}
    n, _, out["dtm"] = ctx.state()
    if ctx.precision == FP64:
        out["n"] = n
    return out


def _mirror(state):
    """The parcels copied into the host's arrays."""
    ctx, arrays = state["ctx"], state["mirror"]
    ptrs = (ctypes.c_void_p * len(arrays))(*[arrays[k].ctypes.data for k in lib.PARCEL_FIELDS])
    st = ctx.L.pmpic_get_parcels(ctx.h, ctypes.byref(ctypes.c_int64()), ptrs)
    if st != 0:
        raise lib.PmpicError(st, "pmpic_get_parcels")
    return arrays


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "ensemble":
        lib.step_concurrent(state["ctxs"], case["steps"])
        return [{k: _kept(c, k) for k in VELOCITY} for c in state["ctxs"]]
    ctx = state["ctx"]
    if kind == "step":
        ctx.step(case["steps"])
        return _look(ctx)
    if kind == "components":
        for _ in range(case["steps"]):
            for _stage in range(4):
                ctx.vort2vel()
                ctx.vorticity_tendency()
                ctx.rk4_integrator()
                ctx.parcel_splitting()
                ctx.parcel_mixing()
        return dict(parcels=_mirror(state), **_look(ctx))
    if kind == "restart":
        ctx.set_time(0.0, case["dt"])
        ctx.set_parcels(state["parcels"])
        ctx.step(case["steps"])
        return dict(parcels=_mirror(state), counts=list(ctx.last_counts()), **_look(ctx))
    if kind == "dump":
        ctx.writebinary_grids()
        return {k: _kept(ctx, k) for k in DUMP}
    if kind == "operators":
        grid = ctx.par2grid(state["var"])
        spec = ctx.fft_forward(grid)
        lap = ctx.laplinv(spec, False)
        ddz = ctx.diffz(lap)
        back = ctx.fft_backward(ddz)
        return dict(grid=grid, spec=spec, lap=lap, ddz=ddz, back=back, par=ctx.grid2par(back))
    st = ctx.L.pmpic_par2grid_noalloc(ctx.h, ctypes.c_void_p(state["var"].data_ptr()),
                                      ctypes.c_void_p(state["out"].data_ptr()))
    if st != 0:
        raise lib.PmpicError(st, "pmpic_par2grid_noalloc")
    return state["out"]


def work(case):
    """Bytes that must cross memory and operations of one pass.  A timestep of the FP64 form moves
    the parcel state of its four stages once in and once out (1248 B a parcel), the FP32-bulk
    form 644 B: offsets, cell, vorticity and the RK4 arrays read and written by each stage, the
    eight fields each par2grid and the mixing read.  Per node and stage: four grids made from
    the parcels, nine velocity, vorticity and tendency grids made from those and six gathered."""
    if case["kind"] == "ensemble":
        parts = [work(dict(m, steps=case["steps"])) for m in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    nx, ny, nz, w = case["nx"], case["ny"], case["nz"] + 1, 4 if case["precision"] == FP32 else 8
    nodes, n = nx * ny * nz, nx * ny * case["nz"] * case["ppc"] ** 3
    halo = (nx + 4) * (ny + 4) * nz * 8
    fft = 2.5 * nodes * math.log2(nx * ny)  # one real 2-D transform of every level
    if case["kind"] in ("step", "components", "restart"):
        bytes_ = case["steps"] * (n * (644 if w == 4 else 1248) + 4 * nodes * 19 * w) + 3 * halo
        bytes_ += {"restart": 2, "components": 1, "step": 0}[case["kind"]] * 17 * 8 * n
        return {"bytes": bytes_, "flops": case["steps"] * 4 * (n * 300 + 18 * fft + 200 * nodes)}
    if case["kind"] == "dump":
        return {"bytes": n * 9 * w + 10 * (nodes * w + halo), "flops": n * 120}
    if case["kind"] == "operators":
        return {"bytes": n * 7 * 8 + 2 * n * 8 + 8 * halo + 8 * nodes * 8,
                "flops": n * 80 + 2 * fft + 40 * nodes}
    return {"bytes": n * 5 * 8 + halo, "flops": n * 40}


# ---- the same results in 64 bits, in plain torch ----------------------------------------------
class _Model:
    """One PMPIC run in FP64: par2grid, the semi-spectral inversion, RK4 (no events)."""

    def __init__(self, case, parcels):
        self.nx, self.ny, self.nz = case["nx"], case["ny"], case["nz"] + 1
        self.dx, self.dy, self.dz = LX / self.nx, LX / self.ny, LZ / case["nz"]
        self.p = {k: torch.as_tensor(v, dtype=torch.float64) for k, v in parcels.items()}
        self.dev = self.p["x"].device
        self.dt = self.dtmax = case.get("dt", 0.01)
        self.fy, self.by, my = self._dft(self.ny, LX)
        self.fx, self.bx, mx = self._dft(self.nx, LX)
        self.kx = 2 * math.pi * mx[None, None, :].expand(1, len(my), len(mx))
        self.ky = 2 * math.pi * my[None, :, None].expand(1, len(my), len(mx))
        kk = my[:, None] ** 2 + mx[None, :] ** 2
        self.k2 = kk * (2 * math.pi) ** 2
        self.keep = (kk <= ((self.nx / 2 / LX) ** 2 + (self.ny / 2 / LX) ** 2) * 2 / 9).double()
        f = self._f32
        nz, dz = self.nz, self.dz
        # the compact z derivative: A out = B f (+ boundary terms), as one matrix per form
        a = torch.eye(nz, dtype=torch.float64) * f(2 / 3)
        rhs = torch.zeros(nz, nz, dtype=torch.float64)
        for k in range(1, nz - 1):
            a[k, k - 1] = a[k, k + 1] = f(1 / 6)
            rhs[k, k + 1], rhs[k, k - 1] = 0.5 / dz, -0.5 / dz
        a[0, 0] = a[-1, -1] = 1.0
        self.dz_free = torch.linalg.solve(a, rhs).to(self.dev)
        a2, rhs2 = a.clone(), rhs.clone()
        a2[0, 1] = a2[-1, -2] = f(1 / 3)
        rhs2[0, 1], rhs2[-1, -2] = 1 / dz, -1 / dz
        rhs2[0, 0] += -f(1 / 6) * dz
        rhs2[-1, -1] += f(1 / 6) * dz
        self.dz_bound = a2, rhs2

    @staticmethod
    def _f32(v):
        return float(np.float32(v))

    def _dft(self, n, length):
        """Real transform of a row to interleaved (Re, Im) of n // 2 + 1 modes, and back."""
        m = torch.arange(n // 2 + 1, dtype=torch.float64, device=self.dev)
        j = torch.arange(n, dtype=torch.float64, device=self.dev)
        ang = torch.remainder(m[:, None] * j[None, :], n) * (2 * math.pi / n)
        fwd = torch.stack((torch.cos(ang), -torch.sin(ang)), 1).reshape(-1, n)
        w = torch.full((n // 2 + 1, 1), 2.0 / n, dtype=torch.float64, device=self.dev)
        w[0] = 1.0 / n
        real = torch.zeros(n // 2 + 1, dtype=torch.bool, device=self.dev)
        real[0] = True
        if n % 2 == 0:
            w[-1], real[-1] = 1.0 / n, True
        s = torch.where(real[:, None], torch.zeros_like(ang), -w * torch.sin(ang))
        bwd = torch.stack((w * torch.cos(ang), s), 1).reshape(-1, n)
        return fwd, bwd.t().contiguous(), torch.repeat_interleave(m, 2) / length

    def forward(self, g):
        t = g.reshape(-1, self.nx) @ self.fx.t()
        t = t.reshape(self.nz, self.ny, -1).transpose(1, 2).reshape(-1, self.ny) @ self.fy.t()
        return t.reshape(self.nz, self.fx.shape[0], -1).transpose(1, 2).contiguous()

    def backward(self, s):
        t = s.reshape(-1, s.shape[2]) @ self.bx.t()
        t = t.reshape(self.nz, s.shape[1], self.nx).transpose(1, 2).reshape(-1, s.shape[1])
        t = t @ self.by.t()
        return t.reshape(self.nz, self.nx, self.ny).transpose(1, 2).contiguous()

    def ddx(self, s):
        out = torch.empty_like(s)
        out[:, :, 0::2], out[:, :, 1::2] = -s[:, :, 1::2], s[:, :, 0::2]
        return out * self.kx

    def ddy(self, s):
        out = torch.empty_like(s)
        out[:, 0::2], out[:, 1::2] = -s[:, 1::2], s[:, 0::2]
        return out * self.ky

    def ddz(self, s):
        return (self.dz_free @ s.reshape(self.nz, -1)).reshape(s.shape)

    def ddz_bound(self, s, bot, top):
        a, rhs = self.dz_bound
        r = rhs.clone()
        dz16 = self._f32(1 / 6) * self.dz
        r[0, 0] += dz16  # the boundary terms take the planes given, not the column's own ends
        r[-1, -1] -= dz16
        d = (r.to(self.dev) @ s.reshape(self.nz, -1)).reshape(s.shape)
        d[0] -= dz16 * bot
        d[-1] += dz16 * top
        return (torch.linalg.inv(a).to(self.dev) @ d.reshape(self.nz, -1)).reshape(s.shape)

    def laplinv(self, s, df0):
        """The compact inverse Laplacian of every column; the k = 0 columns are left alone."""
        f, nz = self._f32, self.nz
        i2, k2 = 1 / self.dz ** 2, self.k2
        off, mid = i2 - f(1 / 12) * k2, -2 * i2 - f(5 / 6) * k2
        d = torch.zeros_like(s)
        d[1:-1] = f(1 / 12) * (s[:-2] + s[2:]) + f(5 / 6) * s[1:-1]
        zero, one = torch.zeros_like(k2), torch.ones_like(k2)
        if df0:
            bend, cend = -i2 - f(1 / 3) * k2, i2 - f(1 / 6) * k2
            d[0] = f(1 / 3) * s[0] + f(1 / 6) * s[1]
            d[-1] = f(1 / 3) * s[-1] + f(1 / 6) * s[-2]
        else:
            bend, cend = one, zero
        skip = k2 == 0
        cp, den = [], torch.where(skip, one, bend)
        d[0] = d[0] / den
        c = cend
        for k in range(1, nz):
            a, b = (off, mid) if k < nz - 1 else (cend, bend)
            cp.append(c / den)
            den = torch.where(skip, one, b - a * cp[-1])
            d[k] = (d[k] - a * d[k - 1]) / den
            c = off
        for k in range(nz - 2, -1, -1):
            d[k] = d[k] - cp[k] * d[k + 1]
        return torch.where(skip, s, d)

    def corners(self):
        """Node and weight of every parcel's eight corners."""
        p, out = self.p, []
        u, v, w = p["x"] / self.dx, p["y"] / self.dy, p["z"] / self.dz
        i, j, k = u.floor(), v.floor(), w.floor().clamp_(max=self.nz - 2)
        ox, oy, oz = u - i, v - j, w - k
        i, j, k = i.long(), j.long(), k.long()
        for c in range(8):
            a, b, e = c & 1, c >> 1 & 1, c >> 2
            node = ((k + e) * self.ny + (j + b) % self.ny) * self.nx + (i + a) % self.nx
            out.append((node, (oz if e else 1 - oz) * (oy if b else 1 - oy) *
                        (ox if a else 1 - ox)))
        return out

    def par2grid(self, fields):
        at = self.corners()
        sums = torch.zeros(len(fields) + 1, self.nz * self.ny * self.nx, dtype=torch.float64,
                           device=self.dev)
        for node, w in at:
            wv = w * self.p["vol"]
            sums[0].index_add_(0, node, wv)
            for f, v in enumerate(fields):
                sums[f + 1].index_add_(0, node, wv * v)
        den = torch.where(sums[0] == 0, torch.ones_like(sums[0]), sums[0])
        return [(s / den).reshape(self.nz, self.ny, self.nx) for s in sums[1:]]

    def tendencies(self, first):
        p, f = self.p, self._f32
        hl = p["h"] - torch.exp(-p["z"])
        P, Q, R, B = self.par2grid([p["p"], p["q"], p["r"], p["b"] + 12.5 * hl.clamp(min=0)])
        a, b, c = self.forward(P), self.forward(Q), self.forward(R)
        cz = torch.empty_like(c)
        cz[1:-1] = (c[2:] - c[:-2]) / 2 / self.dz
        cz[0] = (4 * c[1] - c[2] - 3 * c[0]) / 2 / self.dz
        cz[-1] = (c[-3] + 3 * c[-1] - 4 * c[-2]) / 2 / self.dz
        div = self.ddx(a) + self.ddy(b) + cz
        div[:, 0, 0] = 0
        phi = self.laplinv(div, True) * self.keep
        a, b, c = a - self.ddx(phi), b - self.ddy(phi), c - self.ddz(phi)
        c[0] = 0
        self.P, self.Q, self.R = (self.backward(s * self.keep) for s in (a, b, c))
        da, db = (a * self.keep)[:, 0, 0], (b * self.keep)[:, 0, 0]
        zero = torch.zeros(1, dtype=torch.float64, device=self.dev)
        ubar = torch.cat((zero, torch.cumsum(self.dz / 2 * (db[:-1] + db[1:]), 0)))
        vbar = torch.cat((zero, -torch.cumsum(self.dz / 2 * (da[:-1] + da[1:]), 0)))
        for m in (ubar, vbar):
            m -= f(1 / np.float32(self.nz)) * (m[:-1] + 0.5 * m[-1]).sum()
        ta, tb = a, b
        a, b, c = self.laplinv(a, False), self.laplinv(b, False), self.laplinv(c, True)
        u = self.ddz_bound(b, tb[0], tb[-1]) - self.ddy(c)
        v = self.ddx(c) - self.ddz_bound(a, ta[0], ta[-1])
        u[:, 0, 0], v[:, 0, 0] = ubar, vbar
        w = self.ddy(a) - self.ddx(b)
        self.U, self.V, self.W = (self.backward(s) for s in (u, v, w))
        u, v, w, bs = u * self.keep, v * self.keep, w * self.keep, self.forward(B)
        back = self.backward
        dudx, dvdy = back(self.ddx(u)), back(self.ddy(v))
        dwdx, dwdy = back(self.ddx(w)), back(self.ddy(w))
        P, Q, R = self.P, self.Q, self.R
        dp = back(self.ddy(bs)) + P * dudx + Q * back(self.ddy(u)) + R * (Q + dwdx)
        dq = -back(self.ddx(bs)) + P * back(self.ddx(v)) + Q * dvdy + R * (dwdy - P)
        dr = P * dwdx + Q * dwdy - R * dudx - R * dvdy
        if first:
            tiny = self._f32(1e-15)
            lim = [length / max(float(g.abs().max()), tiny) for g, length in
                   ((self.U, LX), (self.V, LX), (self.W, self.nz * self.dz))]
            om = float((P * P + Q * Q + R * R).max()) ** 0.5
            self.dt = min([self.dtmax] + lim + ([0.5 / om] if om > 0 else []))
        at, grids = self.corners(), [self.U, self.V, self.W, dp, dq, dr]
        return [sum(w * g.reshape(-1)[node] for node, w in at) for g in grids]

    def step(self):
        """One timestep; False when a parcel splits or the mixing would act."""
        p, names = self.p, ("x", "y", "z", "p", "q", "r")
        old = [p[k].clone() for k in names]
        acc = [t.clone() for t in old]
        for stage, (share, move) in enumerate(((6, 0.5), (3, 0.5), (3, 1.0), (6, None))):
            kv = self.tendencies(stage == 0)
            for f, k in enumerate(names):
                acc[f] += self.dt / share * kv[f]
                p[k] = (old[f] + move * self.dt * kv[f]) if move else acc[f].clone()
            z = p["z"].abs()
            p["z"] = torch.where(z > LZ, 2 * LZ - z, z)
            p["x"], p["y"] = torch.remainder(p["x"], LX), torch.remainder(p["y"], LX)
        ds = sum(p[k] * kv[3 + f] for f, k in enumerate(("p", "q", "r"))).abs()
        p["stretch"] = p.get("stretch", torch.zeros_like(ds)) + ds ** self._f32(1 / 3) * self.dt
        cell = ((p["z"] / self.dz).floor().clamp_(max=self.nz - 2) * self.ny +
                (p["y"] / self.dy).floor()) * self.nx + (p["x"] / self.dx).floor()
        fill = torch.bincount(cell.long(), minlength=(self.nz - 1) * self.ny * self.nx)
        vmin = self.dx * self.dy * self.dz / 216
        return not (bool((p["stretch"] > 4).any()) or int(fill.min()) < 3 or
                    bool((p["vol"] < vmin).any()))

    def halo(self, g):
        g = torch.nn.functional.pad(g[None], (2, 2, 2, 2), mode="circular")[0]
        return g.permute(2, 1, 0).contiguous()


def exact(case, seed):
    if case["kind"] in ("ensemble", "restart"):
        return None  # many members; a run of threshold events, whose order is the result
    n = case["nx"] * case["ny"] * case["nz"] * case["ppc"] ** 3
    if n * (4 * case["steps"] if case["kind"] in ("step", "components") else 1) > 400_000_000:
        return None
    parcels = _of(case, seed)
    model = _Model(case, parcels)
    if case["kind"] in ("step", "components"):
        for s in range(case["steps"]):
            if not model.step() and s + 1 < case["steps"]:
                return None
        out = {k: model.halo(g) for k, g in zip(VELOCITY, (model.U, model.V, model.W))}
        return dict(out, dtm=model.dt)
    if case["kind"] == "dump":
        if not model.step():
            return None
        p = model.p
        out = {k: model.halo(g) for k, g in zip(VELOCITY, (model.U, model.V, model.W))}
        vol = torch.zeros(model.nz * model.ny * model.nx, dtype=torch.float64, device=model.dev)
        for node, w in model.corners():
            vol.index_add_(0, node, w * p["vol"])
        vol = vol.reshape(model.nz, model.ny, model.nx)
        vol[0], vol[-1] = 2 * vol[0], 2 * vol[-1]
        b, hg, P, Q, R = model.par2grid([p[k] for k in ("b", "h", "p", "q", "r")])
        z = torch.arange(model.nz, dtype=torch.float64, device=model.dev)[:, None, None] * model.dz
        liq = (hg - torch.exp(-z)).clamp(min=0)
        rest = dict(p=P, q=Q, r=R, b=b + 12.5 * liq, hg=hg, hgliq=liq, vol=vol)
        return dict(out, **{k: model.halo(g) for k, g in rest.items()})
    grid, = model.par2grid([parcels["b"]])
    if case["kind"] == "noalloc":
        return model.halo(grid)
    spec = model.forward(grid)
    lap = model.laplinv(spec, False)
    ddz = model.ddz(lap)
    back = model.backward(ddz)
    par = sum(w * back.reshape(-1)[node] for node, w in model.corners())
    return dict(grid=model.halo(grid), back=model.halo(back), par=par,
                **{k: s.permute(2, 1, 0).contiguous()
                   for k, s in (("spec", spec), ("lap", lap), ("ddz", ddz))})
