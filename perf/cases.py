"""The work that users of this engine have it do, as measurable cases.

Every case is one operator call on one padded grid (or one batch of windows),
through the entry points a program uses: ``_capi.Context`` and ``_capi.Batch``
with arrays on the GPU or on the host, and the autograd operator of ``fwi``.
Grids, time axes and shot counts span those of the repository's workloads
(``workloads.py``), benchmark and tests: 200 x 400 to 1000 x 3000 model points
at 10 m with a 50-point sponge, 15 Hz Ricker sources and a receiver line at
20 m depth, 2 or 4 fine steps per coarse sample.  The time axes are cut so
that a pass stays below a second; the work per time step is that of the full
ones.

``exact`` restates each operator in 64 bits with dense derivative matrices in
plain torch: no kernel, no tiling, nothing of the engine.
"""
import math

import numpy as np
import torch

from acoustic_isotropic_operators_amd import _capi as A
from acoustic_isotropic_operators_amd.fwi import NonlinearVelocityOperator

FAT, PAD, D = 5, 50, 10.0          # stencil ring, sponge width, grid spacing in m
ALPHA, F0, T0, FMAX = 0.95, 15.0, 0.1, 37.5

# propagations per shot of each kind (the gradient's checkpointed
# recomputation is the engine's choice and not counted)
PROPS = dict(nl_fwd=1, nl_adj=1, born_fwd=2, born_adj=2, ext_fwd=2, ext_adj=2, tomo_fwd=5, tomo_adj=4, wemva_fwd=4,
             wemva_adj=4, fwi=3, windows=1)


def _case(name, kind, nz, nx, nts, shots, sub=2, ext="none", next_=1, fs=False, host=False):
    c = dict(kind=kind, nz=nz, nx=nx, nts=nts, shots=shots, sub=sub, ext=ext, next=next_, fs=fs, host=host)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one shot modeled on the smallest grid, host arrays in and out, as the
        # drop-in operator layer calls it: bound by launches
        _case("model_one_small_shot", "nl_fwd", 200, 400, 1000, 1, sub=4, host=True),
        # sources back-propagated for a short line on an odd grid
        _case("model_adjoint_line", "nl_adj", 287, 653, 600, 6),
        # least-squares migration: linearized modeling of a line...
        _case("born_forward_line", "born_fwd", 500, 1200, 1000, 24),
        # ...and its migration, the source wavefield kept in memory
        _case("born_adjoint_line", "born_adj", 500, 1200, 600, 20),
        # linearized modeling with 4 fine steps per sample on a small model
        _case("born_forward_sub4", "born_fwd", 200, 400, 400, 6, sub=4),
        # migration under a free surface
        _case("born_adjoint_surface", "born_adj", 311, 777, 500, 8, fs=True),
        # extended migration, 21 subsurface offsets: modeling and imaging
        _case("offset_forward", "ext_fwd", 500, 1200, 800, 6, ext="offset", next_=21),
        _case("offset_adjoint", "ext_adj", 400, 1000, 400, 10, ext="offset", next_=21),
        # the same with 21 time lags
        _case("lag_adjoint", "ext_adj", 333, 871, 400, 8, ext="time", next_=21),
        # tomographic velocity update from extended data
        _case("tomo_adjoint", "tomo_adj", 300, 700, 300, 6, ext="offset", next_=21),
        # one full-waveform inversion iteration: misfit and its gradient
        _case("fwi_misfit_gradient", "fwi", 400, 1000, 800, 8),
        # many shots on apertures of uneven width, advanced together
        _case("windows_uneven", "windows", 400, 1500, 800, 24),
    ]


def _steps(c):
    return (c["nts"] - 1) * c["sub"]


def _interior(c, nx=None):
    up = lambda n: -(-n // 16) * 16  # noqa: E731
    return up(c["nz"] + (PAD if c["fs"] else 2 * PAD)), up((nx or c["nx"]) + 2 * PAD)


def _updates(c):
    if c["kind"] == "windows":
        pts = sum(math.prod(_interior(c, w)) for w in _widths(c))
    else:
        pts = math.prod(_interior(c)) * c["shots"]
    return pts * _steps(c) * PROPS[c["kind"]]


def draw(rng):
    kinds = ["nl_fwd", "nl_adj", "born_fwd", "born_fwd", "born_adj", "born_adj", "ext_fwd", "ext_adj", "tomo_fwd",
             "tomo_adj", "wemva_fwd", "wemva_adj", "fwi", "windows"]
    while True:
        kind = rng.choice(kinds)
        extended = kind.startswith(("ext", "tomo", "wemva"))
        c = _case(None, kind, nz=int(round(math.exp(rng.uniform(math.log(120), math.log(1000))))),
                  nx=int(round(math.exp(rng.uniform(math.log(250), math.log(3000))))),
                  nts=int(round(math.exp(rng.uniform(math.log(150), math.log(1500))))),
                  shots=int(round(math.exp(rng.uniform(0, math.log(40))))), sub=rng.choice([2, 2, 2, 3, 4]),
                  ext=rng.choice(["offset", "offset", "time"]) if extended else "none",
                  next_=rng.choice([5, 11, 21, 21, 31]) if extended else 1,
                  fs=not kind.startswith(("wemva", "fwi", "windows")) and rng.random() < 0.2,
                  host=kind != "windows" and rng.random() < 0.3)
        if kind == "windows":
            c["nx"] = max(c["nx"], 600)
        if c["ext"] == "time" and c["nts"] < 2 * c["next"]:
            continue
        # modeled reflections need a record that is long enough for them
        if kind in ("born_fwd", "ext_fwd", "tomo_fwd") and c["nts"] * _dts(c) < 0.4 + 0.0025 * c["nz"]:
            continue
        # no more work or memory than the largest listed case has
        nzi, nxi = _interior(c)
        slices = c["nts"] * (2 if kind.startswith(("tomo", "wemva")) else 1) if PROPS[kind] > 1 and kind != "fwi" else 4
        if c["ext"] != "none":
            slices += 40 + c["next"]
        cost = _updates(c) * (1.6 if extended else 1.0)
        if 2e8 < cost < 6e10 and slices * c["shots"] * nzi * nxi * 4 < 2.5e10:
            return c


def work(c):
    """Inputs read once and outputs written once; one update is 33 operations
    of the Laplacian and 5 of the step."""
    nzi, nxi = _interior(c)
    pts, traces = (nzi + 2 * FAT) * (nxi + 2 * FAT), c["shots"] * c["nx"] * c["nts"]
    models = {"ext_fwd": c["next"], "ext_adj": c["next"], "tomo_fwd": 1 + c["next"], "tomo_adj": 1 + c["next"],
              "wemva_fwd": 1 + c["next"], "wemva_adj": 1 + c["next"], "fwi": 2, "born_fwd": 1, "born_adj": 1}
    if c["kind"] == "windows":
        w = _widths(c)
        pts, traces = sum((nzi + 2 * FAT) * (_interior(c, x)[1] + 2 * FAT) for x in w), sum(w) * c["nts"]
    return {"bytes": 4.0 * (pts * (1 + models.get(c["kind"], 0)) + traces), "flops": 38.0 * _updates(c)}


# ------------------------------------------------------------------- inputs --
def _widths(c):
    """Aperture widths of the windows, uneven between a fifth and all of nx."""
    k = np.arange(c["shots"])
    return [int(c["nx"] * (0.2 + 0.8 * ((0.618034 * (i + 1)) % 1.0))) for i in k]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _smooth_noise(g, nx, nz, cell):
    """Random field varying over about `cell` points, within [-1, 1]."""
    coarse = torch.rand((1, 1, nx // cell + 4, nz // cell + 4), generator=g, device="cuda") * 2 - 1
    f = torch.nn.functional.interpolate(coarse, size=(nx, nz), mode="bicubic", align_corners=True)[0, 0]
    return f.clamp(-1, 1)


def _pad(c, m, nx, zero=False):
    """The physical [nx][nz] model on the padded grid: edges repeated (or zero)
    outside it, the stencil ring zero."""
    nzi, nxi = _interior(c, nx)
    top = 0 if c["fs"] else PAD
    size = (PAD, nxi - PAD - nx, top, nzi - top - m.shape[1])
    p = torch.nn.functional.pad(m[None, None], (size[2], size[3], size[0], size[1]),
                                mode="constant" if zero else "replicate")[0, 0]
    return torch.nn.functional.pad(p, (FAT, FAT, FAT, FAT)).contiguous()


def _velocity(c, g, nx):
    z = torch.linspace(0, 1, c["nz"], device="cuda")
    vmax = 4000.0 if c["kind"] != "fwi" else 4200.0
    return (1500.0 + (vmax - 1500.0) * z) * (1.0 + 0.05 * _smooth_noise(g, nx, c["nz"], 30))


def _reflectivity(c, g, nx):
    """Random spikes along dipping interfaces."""
    m = torch.zeros((nx, c["nz"]), device="cuda")
    x = torch.arange(nx, device="cuda")
    for _ in range(10):
        r = torch.rand(2, generator=g, device="cuda")
        zi = ((0.15 + 0.8 * r[0]) * c["nz"] + 0.3 * (r[1] - 0.5) * (x - nx / 2)).round().long().clamp(0, c["nz"] - 1)
        keep = torch.rand(nx, generator=g, device="cuda") < 0.5
        m[x, zi] = torch.where(keep, torch.randn(nx, generator=g, device="cuda"), m[x, zi])
    return m


def _ricker(c):
    t = np.arange(c["nts"]) * _dts(c) - T0
    a = (np.pi * F0 * t) ** 2
    return ((1.0 - 2.0 * a) * np.exp(-a)).astype(np.float32)


def _dts(c):
    return 0.001 if c["kind"] == "fwi" else 0.001 * c["sub"]


def _gathers(c, g, xs):
    """Shot gathers [shots][nx][nts]: reflections with moveout, and noise."""
    S, nx, nts = c["shots"], c["nx"], c["nts"]
    off = (torch.arange(nx, device="cuda")[None] - torch.tensor(xs, device="cuda")[:, None]).float() * D
    t = torch.arange(nts, device="cuda").float() * _dts(c)
    out = 0.05 * torch.randn((S, nx, nts), generator=g, device="cuda")
    for _ in range(6):
        r = torch.rand(3, generator=g, device="cuda")
        t0, v = 0.1 + r[0] * 0.8 * nts * _dts(c), 1800.0 + 1500.0 * r[1]
        tau = torch.sqrt(t0 * t0 + (off / v) ** 2)
        a = (math.pi * F0 * (t[None, None] - tau[..., None])) ** 2
        out += (r[2] - 0.5) * (1 - 2 * a) * torch.exp(-a)
    return out


def _params(c, nx):
    nzi, nxi = _interior(c, nx)
    top = 0 if c["fs"] else PAD
    ext = dict(none=A.EXT_NONE, offset=A.EXT_OFFSET, time=A.EXT_TIME)[c["ext"]]
    return dict(nz=nzi + 2 * FAT, nx=nxi + 2 * FAT, dz=D, dx=D, nts=c["nts"], dts=_dts(c), sub=c["sub"], zPadMinus=top,
                zPadPlus=nzi - top - c["nz"], xPadMinus=PAD, xPadPlus=nxi - PAD - nx, alphaCos=ALPHA, fMax=FMAX,
                freeSurface=int(c["fs"]), nExt=c["next"], extension=ext)


def _depth(c):
    return FAT + (0 if c["fs"] else PAD) + 2


def _source_columns(c):
    return [int((k + 0.5) * c["nx"] / c["shots"]) for k in range(c["shots"])]


def _inputs(c, seed):
    """What both the engine and `exact` start from, on the padded grid."""
    g = _gen(seed)
    x = dict(vel=_pad(c, _velocity(c, g, c["nx"]), c["nx"]), wav=_ricker(c), xs=_source_columns(c))
    # a wavelet of its own for every seed
    x["wav"] = (x["wav"] * np.float32(0.5 + torch.rand(1, generator=g, device="cuda").item())).astype(np.float32)
    k = c["kind"]
    if k.startswith(("born", "tomo", "wemva")):
        x["model"] = _pad(c, _reflectivity(c, g, c["nx"]), c["nx"], zero=True)
    if k.startswith(("tomo", "wemva")):   # a velocity perturbation instead
        x["model"] = _pad(c, 50.0 * _smooth_noise(g, c["nx"], c["nz"], 20), c["nx"], zero=True)
    if k.startswith(("ext", "tomo", "wemva")):   # energy around zero extension, as focused images have
        h = (c["next"] - 1) // 2
        refl = _pad(c, _reflectivity(c, g, c["nx"]), c["nx"], zero=True)
        roll = torch.exp(-(torch.arange(-h, h + 1, device="cuda").float() / (0.3 * h + 1)) ** 2)
        x["ext"] = (roll[:, None, None] * refl).contiguous()
    if k in ("nl_adj", "born_adj", "ext_adj", "tomo_adj", "wemva_fwd", "wemva_adj", "fwi"):
        x["data"] = _gathers(c, g, x["xs"])
    return x


def prepare(c, seed):
    if c["kind"] == "windows":
        return _prepare_windows(c, seed)
    x = _inputs(c, seed)
    p = _params(c, c["nx"])
    S, nts = c["shots"], c["nts"]
    grid = (p["nz"], p["nx"], nts)
    iz = _depth(c)
    src = [(1, iz, 1, 1, FAT + PAD + xs, 1) for xs in x["xs"]]
    rec = (1, iz, 1, c["nx"], FAT + PAD, 1)
    put = (lambda t: t.cpu().numpy()) if c["host"] else (lambda t: t)
    s = dict(c=c, mem=A.MEM_HOST if c["host"] else A.MEM_DEVICE)
    if c["kind"] == "fwi":
        dev = (lambda t: t.cpu()) if c["host"] else (lambda t: t)
        s["op"] = NonlinearVelocityOperator(p, [("grid", a) for a in src], [("grid", rec)], x["wav"][None, None])
        # the observed data at the amplitude of the modeled ones
        s["vel"], s["obs"] = dev(x["vel"]), dev(x["data"] * 0.05)
        return s
    s["ctx"] = A.Context(p)
    s["ctx"].set_velocity(put(x["vel"]), s["mem"])
    s["src"] = [A.Device.grid(*a, *grid) for a in src]
    s["rec"] = [A.Device.grid(*rec, *grid)]
    s["wav"] = x["wav"][None]
    new = lambda *shape: put(torch.zeros(shape, device="cuda"))  # noqa: E731
    k = c["kind"]
    if k == "nl_fwd":
        s["model"], s["out"] = put(torch.from_numpy(x["wav"])[None, None].cuda()), new(S, c["nx"], nts)
    elif k == "nl_adj":
        s["data"], s["out"] = put(x["data"]), new(S, 1, nts)
    elif k in ("born_fwd", "tomo_fwd"):
        s["model"], s["out"] = put(x["model"]), new(S, c["nx"], nts)
    elif k == "ext_fwd":
        s["model"], s["out"] = put(x["ext"]), new(S, c["nx"], nts)
    elif k in ("born_adj", "tomo_adj"):
        s["data"], s["out"] = put(x["data"]), new(p["nx"], p["nz"])
    elif k == "ext_adj":
        s["data"], s["out"] = put(x["data"]), new(c["next"], p["nx"], p["nz"])
    elif k == "wemva_fwd":
        s["data"], s["model"], s["out"] = put(x["data"]), put(x["model"]), new(c["next"], p["nx"], p["nz"])
    elif k == "wemva_adj":
        s["data"], s["image"], s["out"] = put(x["data"]), put(x["ext"]), new(p["nx"], p["nz"])
    if k.startswith("tomo"):
        s["ctx"].set_ext_reflectivity(put(x["ext"]), s["mem"])
    return s


def _window_inputs(c, seed):
    g = _gen(seed)
    full = _velocity(c, g, c["nx"])
    w = _widths(c)
    x0 = [int((c["nx"] - n) * ((0.754878 * (i + 1)) % 1.0)) for i, n in enumerate(w)]
    vels = [_pad(c, full[a:a + n], n) for a, n in zip(x0, w)]
    return vels, w, _ricker(c) * np.float32(0.5 + torch.rand(1, generator=g, device="cuda").item())


def _prepare_windows(c, seed):
    vels, w, wav = _window_inputs(c, seed)
    iz, nts = _depth(c), c["nts"]
    src = [A.Device.grid(1, iz, 1, 1, FAT + PAD + n // 2, 1, v.shape[1], v.shape[0], nts) for v, n in zip(vels, w)]
    rec = [A.Device.grid(1, iz, 1, n, FAT + PAD, 1, v.shape[1], v.shape[0], nts) for v, n in zip(vels, w)]
    b = A.Batch(_params(c, w[0]))
    b.set_windows(vels, src, rec, mem=A.MEM_DEVICE)
    return dict(c=c, batch=b, model=[torch.from_numpy(wav)[None].cuda()],
                out=[torch.zeros((n, nts), device="cuda") for n in w])


def run(s):
    k = s["c"]["kind"]
    if k == "windows":
        s["batch"].nl_forward(s["model"], s["out"], mem=A.MEM_DEVICE)
        return s["out"]
    if k == "fwi":
        return s["op"].misfit_and_gradient(s["vel"], s["obs"])
    ctx, geo = s["ctx"], dict(mem=s["mem"])
    if k == "nl_fwd":
        ctx.nl_forward(s["model"], s["out"], s["src"], s["rec"], **geo)
    elif k == "nl_adj":
        ctx.nl_adjoint(s["out"], s["data"], s["src"], s["rec"], **geo)
    elif k == "wemva_fwd":
        ctx.wemva_forward(s["model"], s["out"], s["data"], s["src"], s["wav"], s["rec"], **geo)
    elif k == "wemva_adj":
        ctx.wemva_adjoint(s["out"], s["image"], s["data"], s["src"], s["wav"], s["rec"], **geo)
    elif k.endswith("fwd"):
        fn = dict(born_fwd=ctx.born_forward, ext_fwd=ctx.bornext_forward, tomo_fwd=ctx.tomo_forward)[k]
        fn(s["model"], s["out"], s["src"], s["wav"], s["rec"], **geo)
    else:
        fn = dict(born_adj=ctx.born_adjoint, ext_adj=ctx.bornext_adjoint, tomo_adj=ctx.tomo_adjoint)[k]
        fn(s["out"], s["data"], s["src"], s["wav"], s["rec"], **geo)
    return s["out"]


# --------------------------------------------------------- 64-bit restatement --
COEF = (-2.927222222, 1.666666667, -0.238095238, 0.039682539, -0.004960317, 0.000317460)


class _Fields:
    """Wavefields [shot][x][z] of some shots on the interior of one padded
    grid (the ring around it is zero), and the operators' building blocks."""

    def __init__(self, c, vel, xs, nx):
        self.c, (self.nzi, self.nxi) = c, _interior(c, nx)
        v = vel[FAT:-FAT, FAT:-FAT].double()
        self.v, self.dtw, self.dts = v, _dts(c) / c["sub"], _dts(c)
        self.v2, self.refl = (v * self.dtw) ** 2, 2.0 / v ** 3
        self.Lx, self.Lz = self._lap(self.nxi), self._lap(self.nzi)
        if c["fs"]:   # odd about the surface row, which is zero
            i = torch.arange(self.nzi, device="cuda")
            s = i[:, None] + i[None]
            cf = torch.tensor(COEF, dtype=torch.float64, device="cuda") / D ** 2
            self.Lz = self.Lz - torch.where(s <= 5, cf[s.clamp(max=5)], torch.zeros_like(self.Lz))
            self.Lz[0], self.Lz[:, 0] = 0, 0
        w = min(PAD, self.nxi - PAD - nx, self.nzi - (0 if c["fs"] else PAD) - c["nz"])
        z, x = torch.arange(self.nzi, device="cuda")[None], torch.arange(self.nxi, device="cuda")[:, None]
        dist = torch.minimum(torch.minimum(x, self.nxi - 1 - x), self.nzi - 1 - z)
        if not c["fs"]:
            dist = torch.minimum(dist, z)
        damp = ALPHA + (1 - ALPHA) * torch.cos(math.pi * (w - dist.double()) / w)
        self.damp = torch.where(dist < w, damp, torch.ones_like(damp))
        i = np.arange(c["sub"] + 1) / c["sub"]
        self.scale = 1.0 / math.sqrt(((c["nts"] - 1) * c["sub"] + 1) / c["nts"])
        self.fl, self.fr = (1 - i) * self.scale, i * self.scale
        self.xs = torch.tensor([PAD + x for x in xs], device="cuda")
        self.row, self.rec, self.S = _depth(c) - FAT, slice(PAD, PAD + nx), len(xs)
        self.at = torch.arange(self.S, device="cuda")

    @staticmethod
    def _lap(n):
        i = torch.arange(n, device="cuda")
        k = (i[:, None] - i[None]).abs()
        cf = torch.tensor(COEF, dtype=torch.float64, device="cuda") / D ** 2
        return torch.where(k <= 5, cf[k.clamp(max=5)], torch.zeros((), dtype=torch.float64, device="cuda"))

    def zeros(self, *lead):
        return torch.zeros((*lead, self.nxi, self.nzi), dtype=torch.float64, device="cuda")

    def lap(self, p):
        return torch.matmul(p, self.Lz) + torch.matmul(self.Lx, p)

    def source(self, wav, born):
        """The wavelet at fine steps, scaled at each shot's source point."""
        w = torch.from_numpy(wav).cuda().double()
        if born:
            e = torch.nn.functional.pad(w, (1, 1))
            w = (e[2:] - 2 * w + e[:-2]) / self.dts ** 2
        return self.fine(w)[:, None] * ((self.dtw * self.v[self.xs, self.row]) ** 2)[None]

    def fine(self, w):
        t = torch.arange((self.c["nts"] - 1) * self.c["sub"], device="cuda")
        k, a = t // self.c["sub"], (t % self.c["sub"]).double() / self.c["sub"]
        return (w[k] * (1 - a) + w[k + 1] * a) * self.scale

    def forward(self, sig=None, ss=None, capture=None, record=None, keep=None):
        """Fine steps forward in time: sig [t][shot] at the sources, ss(k) the
        secondary source of coarse sample k; fills capture [k][...] and record."""
        c, o, cur = self.c, self.zeros(self.S), self.zeros(self.S)
        a = ss(0) if ss else None
        for k in range(c["nts"] - 1):
            b = ss(k + 1) if ss else None
            for i in range(1, c["sub"] + 1):
                if c["fs"]:
                    o[..., 0], cz = 0, cur.clone()
                    cz[..., 0] = 0
                else:
                    cz = cur
                n = self.v2 * self.lap(cz) + 2 * cz - o
                if sig is not None:
                    n[self.at, self.xs, self.row] += sig[k * c["sub"] + i - 1]
                if ss:
                    n += a * self.fl[i - 1] + b * self.fr[i - 1]
                n *= self.damp
                if keep is not None:
                    keep[k * c["sub"] + i - 1] = cur      # the slice this step starts from
                o, cur = cur * self.damp, n
                if capture is not None:
                    capture[k] += n * self.fl[i]
                    capture[k + 1] += n * self.fr[i]
                if record is not None:
                    r = n[:, self.rec, self.row]
                    record[:, :, k] += r * self.fl[i]
                    record[:, :, k + 1] += r * self.fr[i]
            a = b

    def backward(self, data=None, ss=None, capture=None, at_source=None, each=None):
        """The adjoint steps, backward in time, driven by data or by ss(k)."""
        c, o, cur = self.c, self.zeros(self.S), self.zeros(self.S)
        b = ss(c["nts"] - 1) if ss else None
        for k in range(c["nts"] - 2, -1, -1):
            a = ss(k) if ss else None
            for i in range(c["sub"] - 1, -1, -1):
                n = self.lap(self.v2 * cur) + 2 * cur - o
                if c["fs"]:
                    n[..., 0] = 0
                if data is not None:
                    n[:, self.rec, self.row] += data[:, :, k] * self.fl[i + 1] + data[:, :, k + 1] * self.fr[i + 1]
                if ss:
                    n += a * self.fl[i + 1] + b * self.fr[i + 1]
                n *= self.damp
                o, cur = cur * self.damp, n
                if capture is not None:
                    capture[k] += n * self.fl[i]
                    capture[k + 1] += n * self.fr[i]
                if at_source is not None:
                    at_source[k * c["sub"] + i] = n[self.at, self.xs, self.row]
                if each:
                    each(k * c["sub"] + i, n)
            b = a

    # the extension's scattering and imaging about the model points x, with
    # offset h or lag l of slice e; dir = -1 swaps the two wavefields' roles
    def pairs(self, k, dir=1):
        c, hx = self.c, (self.c["next"] - 1) // 2
        for e in range(c["next"]):
            h = e - hx
            if c["ext"] == "offset":
                m = slice(hx, self.nxi - hx)
                yield e, m, slice(hx + h, self.nxi - hx + h), slice(hx - h, self.nxi - hx - h), k
            elif 0 <= k - dir * 2 * h < c["nts"]:
                yield e, slice(None), slice(None), slice(None), k - dir * 2 * h

    def scatter(self, m, W):
        def ss(k):
            out = self.zeros(self.S)
            for e, x, r, s, j in self.pairs(k):
                out[:, r] += m[e, x] * W[j][:, s]
            return out * self.v2 if self.c["ext"] == "offset" else out
        return ss

    def scatter_adjoint(self, m, R):
        def ss(k):
            out = self.zeros(self.S)
            for e, x, r, s, j in self.pairs(k, -1):
                f = R[j][:, r] * self.v2[r] if self.c["ext"] == "offset" else R[j]
                out[:, s] += m[e, x] * f
            return out
        return ss

    def image(self, img, W, P, dir=1):
        """img[e] += (receiver side) * (source side); dir = -1: the lag shifts W, here the receiver field."""
        for k in range(self.c["nts"]):
            for e, x, r, s, j in self.pairs(k, dir):
                if self.c["ext"] == "offset":
                    img[e, x] += ((P[k][:, r] * self.v2[r]) * W[j][:, s]).sum(0)
                else:
                    img[e] += (P[k] * W[j]).sum(0)

    def ext_scale(self):
        return self.refl if self.c["ext"] == "offset" else self.refl * self.v2

    def d2(self, W):
        z = torch.zeros_like(W[:1])
        return (torch.cat([W[1:], z]) + torch.cat([z, W[:-1]]) - 2 * W) / self.dts ** 2


def _grow(c, m):
    return torch.nn.functional.pad(m, (FAT, FAT, FAT, FAT))


def _exact_shots(c, x, sel):
    """The operator on the shots `sel`, all at once; a sum over them where the
    operator sums over shots."""
    f = _Fields(c, x["vel"], [x["xs"][i] for i in sel], c["nx"])
    k, nts, S = c["kind"], c["nts"], len(sel)
    cut = lambda m: m[..., FAT:-FAT, FAT:-FAT].double()  # noqa: E731
    data = x["data"][sel].double() if "data" in x else None
    rec = torch.zeros((S, c["nx"], nts), dtype=torch.float64, device="cuda")
    if k == "nl_fwd":
        f.forward(sig=f.source(x["wav"], False), record=rec)
        return rec
    if k == "nl_adj":
        fine = torch.zeros((_steps(c), S), dtype=torch.float64, device="cuda")
        f.backward(data=data, at_source=fine)
        out = torch.zeros((nts, S), dtype=torch.float64, device="cuda")
        for i in range(c["sub"]):
            out[:-1] += fine[i::c["sub"]] * f.fl[i]
            out[1:] += fine[i::c["sub"]] * f.fr[i]
        return (out * ((f.dtw * f.v[f.xs, f.row]) ** 2)).T[:, None].contiguous()
    if k == "fwi":
        T = _steps(c)
        keep = f.zeros(T, S)
        f.forward(sig=f.source(x["wav"], False), record=rec, keep=keep)
        r = rec - (x["data"][sel] * 0.05).double()
        g, u = f.zeros(), f.fine(torch.from_numpy(x["wav"]).cuda().double())

        def each(t, n):
            g.add_((f.lap(keep[t]) * n).sum(0))
            g.index_put_((f.xs, torch.full_like(f.xs, f.row)), n[f.at, f.xs, f.row] * u[t], accumulate=True)
        f.backward(data=r, each=each)
        return [0.5 * (r * r).sum(), _grow(c, g * 2 * f.v * f.dtw ** 2)]
    W = f.zeros(nts, S)
    f.forward(sig=f.source(x["wav"], True), capture=W)
    if k == "born_fwd":
        m = cut(x["model"]) * f.v2 * f.refl
        f.forward(ss=lambda j: m * W[j], record=rec)
        return rec
    if k == "ext_fwd":
        f.forward(ss=f.scatter(cut(x["ext"]) * f.ext_scale(), W), record=rec)
        return rec
    R = f.zeros(nts, S)
    if k in ("born_adj", "ext_adj"):
        f.backward(data=data, capture=R)
        if k == "born_adj":
            return _grow(c, sum((W[j] * R[j]).sum(0) for j in range(nts)) * f.v2 * f.refl)
        img = f.zeros(c["next"])
        f.image(img, W, R)
        return _grow(c, img * f.ext_scale())
    W = f.d2(W)
    m = cut(x["model"]) * f.v2 * f.refl
    e = cut(x["ext"]) * f.ext_scale()
    P = f.zeros(nts, S)
    if k == "tomo_fwd":
        f.forward(ss=f.scatter(e, W), capture=P)
        f.forward(ss=lambda j: m * P[j], record=rec)
        P.zero_()
        f.forward(ss=lambda j: m * W[j], capture=P)
        f.forward(ss=f.scatter(e, P), record=rec)
        return rec
    f.backward(data=data, capture=R)
    if k == "wemva_fwd":
        img = f.zeros(c["next"])
        f.forward(ss=lambda j: m * W[j], capture=P)
        if c["ext"] == "offset":
            f.image(img, P, R)
        else:
            f.image(img, R, P, dir=-1)
        P.zero_()
        f.backward(ss=lambda j: m * R[j], capture=P)
        f.image(img, W, P)
        return _grow(c, img * f.ext_scale())
    f.forward(ss=f.scatter(e, W), capture=P)       # tomo_adj, wemva_adj
    out = sum((P[j] * R[j]).sum(0) for j in range(nts))
    P.zero_()
    f.backward(ss=f.scatter_adjoint(e, R), capture=P)
    out += sum((P[j] * W[j]).sum(0) for j in range(nts))
    return _grow(c, out * f.v2 * f.refl)


def exact(c, seed):
    if _updates(c) > 8e10:
        return None
    if c["kind"] == "windows":
        vels, w, wav = _window_inputs(c, seed)
        out = []
        for v, n in zip(vels, w):
            f = _Fields(c, v, [n // 2], n)
            rec = torch.zeros((1, n, c["nts"]), dtype=torch.float64, device="cuda")
            f.forward(sig=f.source(wav, False), record=rec)
            out.append(rec[0])
        return out
    x = _inputs(c, seed)
    # as many shots at once as 40 GB of stored wavefields allow
    nzi, nxi = _interior(c)
    stored = dict(nl_fwd=8, nl_adj=8, fwi=_steps(c)).get(c["kind"], c["nts"] * (2 if c["kind"].startswith(("born", "ext"))
                                                                                  else 3))
    n = max(1, min(c["shots"], int(4e10 / (8.0 * stored * nzi * nxi))))
    parts = [_exact_shots(c, x, list(range(i, min(i + n, c["shots"])))) for i in range(0, c["shots"], n)]
    if c["kind"] == "fwi":
        return tuple(sum(p[i] for p in parts) for i in range(2))
    if c["kind"] in ("nl_fwd", "nl_adj", "born_fwd", "ext_fwd", "tomo_fwd"):
        return torch.cat(parts)
    return sum(parts)
