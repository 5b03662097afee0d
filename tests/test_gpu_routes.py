"""Each family of step kernels gives the float oracle's bits on a call that
runs it: the choice of kernels is read back from the context.  Four points
per lane without a free surface (modeling of many points, adjoint modeling
with receivers in the stencil ring); one point per lane, whose tile a caller
has set, on one lane and on two; several steps per launch next to its line;
and the general time-lag kernels, which take more than 41 lags."""
import numpy as np
import pytest

from cases import make_case
from oracle import oracle as O

pytestmark = pytest.mark.gpu
FAT = 5
POINT, WIDE, STEPS64 = 0, 1, 4


def _setup(nzi, nxi, shots, sub, nts, iz=None, ix=None, fs=False):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=nzi + 3 * nxi, nz=nzi + 2 * FAT, nx=nxi + 2 * FAT, nShot=shots, nts=nts, sub=sub,
                  dts=0.001 * sub, src_iz=20, shot_dx=max(1, min(12, (nxi - 20) // shots)))
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=nts, dts=c.dts, sub=sub, alphaCos=c.alpha, fMax=20.0,
                         zPadMinus=0 if fs else c.pad, zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad,
                         freeSurface=int(fs)))
    ctx.set_velocity(c.vel)
    g = O.Grid(nz=c.nz, nx=c.nx, nts=nts, sub=sub, minPad=c.pad, dz=c.dz, dx=c.dx, dts=c.dts, alphaCos=c.alpha,
               freeSurface=int(fs))
    if iz is None:
        iz = list(range(FAT, c.nz - FAT, 13)) + [20]
        ix = [FAT + (7 * k) % nxi for k in range(len(iz) - 1)] + [18]
    srcs = [A.Device.grid(*a, c.nz, c.nx, nts) for _, a in c.src_args]
    recs, orec = [A.Device.ints(iz, ix, c.nz, c.nx, nts)], [O.Device.ints(iz, ix, c.nz, c.nx, nts)]
    return c, ctx, g, srcs, recs, c.oracle_sources(), orec


def _modeling(nzi, nxi, shots, sub, nts, forward, adjoint, **kw):
    c, ctx, g, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, sub, nts, **kw)
    rng = np.random.default_rng(2)
    w = rng.standard_normal((shots, 1, nts)).astype(np.float32)
    d = np.zeros((shots, recs[0].nDev, nts), np.float32)
    ctx.nl_forward(w, d, srcs, recs)
    assert ctx.get_option("kernels") == forward
    ref = O.nl_forward(g, c.vel, osrc, orec, w, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    dr = rng.standard_normal(d.shape).astype(np.float32)
    m = np.zeros((shots, 1, nts), np.float32)
    ctx.nl_adjoint(m, dr, srcs, recs)
    assert ctx.get_option("kernels") == adjoint
    ref = O.nl_adjoint(g, c.vel, osrc, orec, dr, shots, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(m, ref)


@pytest.mark.parametrize("nzi,nxi,shots,sub,nts,forward,adjoint", [
    (272, 304, 24, 2, 12, STEPS64, STEPS64),     # 600 workgroups of 64 x 64
    (432, 464, 17, 2, 8, STEPS64, STEPS64),      # 952
    (432, 464, 32, 2, 8, WIDE, POINT),           # 1792, and 6496 of 64 x 16
    (496, 416, 29, 3, 6, WIDE, POINT)])          # 1624, and 6032
def test_modeling_on_both_sides_of_the_lines(nzi, nxi, shots, sub, nts, forward, adjoint):
    _modeling(nzi, nxi, shots, sub, nts, forward, adjoint)


@pytest.mark.parametrize("nzi,nxi,shots,sub", [(112, 80, 3, 3), (176, 112, 9, 2)])
def test_receivers_in_the_stencil_ring(nzi, nxi, shots, sub):
    _modeling(nzi, nxi, shots, sub, 30, POINT, WIDE, iz=[2, 20, nzi + 7, 20],
              ix=[16, 3, nxi // 2, 18])


@pytest.mark.parametrize("sub", [2, 3])
@pytest.mark.parametrize("lanes", [1, 2])
@pytest.mark.parametrize("tile", [3216, 6432, 0])
def test_lanes(lanes, sub, tile):
    """Tile 0: four points per lane, under a free surface."""
    c, ctx, g, srcs, recs, osrc, orec = _setup(80, 96, 5, sub, 40, fs=tile == 0)
    ctx.set_option("lanes", lanes)
    if tile:
        ctx.set_option("tileFwd", tile)
        ctx.set_option("tileAdj", tile)
    kernels = POINT if tile else WIDE
    rng = np.random.default_rng(lanes + sub)
    wav = c.wavelet[None, :].copy()
    m = rng.standard_normal((c.nx, c.nz)).astype(np.float32)
    dr = rng.standard_normal((5, recs[0].nDev, c.nts)).astype(np.float32)
    d = np.zeros_like(dr)
    ctx.nl_forward(wav[None], d, srcs, recs)
    assert ctx.get_option("kernels") == kernels
    np.testing.assert_array_equal(d, O.nl_forward(g, c.vel, osrc, orec, wav[None], "f"))
    ma = np.zeros((5, 1, c.nts), np.float32)
    ctx.nl_adjoint(ma, dr, srcs, recs)
    assert ctx.get_option("kernels") == kernels
    np.testing.assert_array_equal(ma, O.nl_adjoint(g, c.vel, osrc, orec, dr, 5, "f"))
    ctx.born_forward(m, d, srcs, wav, recs)
    assert ctx.get_option("kernels") == kernels
    ref = O.born_forward(g, c.vel, osrc, [wav], orec, m, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    img = np.zeros((c.nx, c.nz), np.float32)
    ctx.born_adjoint(img, dr, srcs, wav, recs)
    assert ctx.get_option("kernels") == kernels
    np.testing.assert_array_equal(img, O.born_adjoint(g, c.vel, osrc, [wav], orec, dr, "f"))


@pytest.mark.parametrize("nExt,nts,batch", [(43, 30, None), (43, 61, 5), (47, 110, 16)])
def test_more_lags_than_the_register_windows_take(nExt, nts, batch):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=nExt + nts, nz=42, nx=58, nShot=2, nts=nts, sub=2, dts=0.002, nExt=nExt, src_iz=14)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=nts, dts=c.dts, sub=2, alphaCos=c.alpha, fMax=20.0,
                         zPadMinus=c.pad, zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad, nExt=nExt,
                         extension=A.EXT_TIME))
    ctx.set_velocity(c.vel)
    if batch is not None:
        ctx.set_option("extBatch", batch)
    srcs = [A.Device.grid(*a, c.nz, c.nx, nts) for _, a in c.src_args]
    recs = [A.Device.grid(*a, c.nz, c.nx, nts) for _, a in c.rec_args]
    wav = c.wavelet[None, :].copy()
    rng = np.random.default_rng(7)
    m = rng.standard_normal((nExt, c.nx, c.nz)).astype(np.float32)
    dr = rng.standard_normal((2, recs[0].nDev, nts)).astype(np.float32)
    args = (c.grid, c.vel, c.oracle_sources(), [wav], c.oracle_receivers())
    d, ext = np.zeros_like(dr), np.zeros_like(m)
    ctx.bornext_forward(m, d, srcs, wav, recs)
    ref = O.borntime_forward(*args, m, 0, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    ctx.bornext_adjoint(ext, dr, srcs, wav, recs)
    np.testing.assert_array_equal(ext, O.borntime_adjoint(*args, dr, 0, "f"))
