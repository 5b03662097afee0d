"""The step kernels with four z-points per lane give the float oracle's results
bit for bit at the edges of their 64 x 16 and 64 x 32 tiles: interior sizes
that leave a remainder of 16, 32 and 48 rows and of 16 columns, a last tile
narrower than the sponge, and shot counts on both sides of the workgroup
counts at which the calls change kernels."""
import numpy as np
import pytest

from cases import make_case
from oracle import oracle as O

pytestmark = pytest.mark.gpu
FAT = 5


def _setup(nzi, nxi, shots, sub, fs, nts):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=nzi + nxi, nz=nzi + 2 * FAT, nx=nxi + 2 * FAT, nShot=shots, nts=nts, sub=sub, dts=0.001 * sub,
                  src_iz=8, shot_dx=max(1, min(12, (nxi - 20) // shots)))
    pads = dict(zPadMinus=0 if fs else c.pad, zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=c.nts, dts=c.dts, sub=c.sub, alphaCos=c.alpha,
                         fMax=20.0, freeSurface=int(fs), **pads))
    ctx.set_velocity(c.vel)
    g = O.Grid(nz=c.nz, nx=c.nx, nts=c.nts, sub=c.sub, minPad=c.pad, dz=c.dz, dx=c.dx, dts=c.dts, alphaCos=c.alpha,
               freeSurface=int(fs))
    iz = list(range(FAT, c.nz - FAT, 13)) + [c.nz - FAT - 1]          # rows of every tile, first and last
    ix = [FAT + (7 * k) % nxi for k in range(len(iz))]
    srcs = [A.Device.grid(*a, c.nz, c.nx, c.nts) for _, a in c.src_args]
    recs = [A.Device.ints(iz, ix, c.nz, c.nx, c.nts)]
    return A, c, ctx, g, srcs, recs, c.oracle_sources(), [O.Device.ints(iz, ix, c.nz, c.nx, c.nts)]


@pytest.mark.parametrize("fs", [False, True])
@pytest.mark.parametrize("nzi,nxi,shots,sub", [(64, 64, 1, 2), (80, 48, 2, 2), (112, 80, 3, 3), (176, 112, 24, 2)])
def test_born_and_adjoint_modeling(nzi, nxi, shots, sub, fs):
    A, c, ctx, g, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, sub, fs, 40)
    rng = np.random.default_rng(5)
    wav = c.wavelet[None, :].copy()
    m = rng.standard_normal((c.nx, c.nz)).astype(np.float32)
    d = np.zeros((shots, recs[0].nDev, c.nts), np.float32)
    ctx.born_forward(m, d, srcs, wav, recs)
    ref = O.born_forward(g, c.vel, osrc, [wav], orec, m, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    dr = rng.standard_normal(d.shape).astype(np.float32)
    img = np.zeros((c.nx, c.nz), np.float32)
    ctx.born_adjoint(img, dr, srcs, wav, recs)
    np.testing.assert_array_equal(img, O.born_adjoint(g, c.vel, osrc, [wav], orec, dr, "f"))
    ma = np.zeros((shots, 1, c.nts), np.float32)
    ctx.nl_adjoint(ma, dr, srcs, recs)
    np.testing.assert_array_equal(ma, O.nl_adjoint(g, c.vel, osrc, orec, dr, shots, "f"))


@pytest.mark.parametrize("nzi,nxi,shots", [(336, 272, 30), (288, 304, 32), (320, 320, 32)])
def test_modeling_of_many_shots(nzi, nxi, shots):
    A, c, ctx, g, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, 2, False, 24)
    w = c.wavelet[None, None, :].copy()
    d = np.zeros((shots, recs[0].nDev, c.nts), np.float32)
    ctx.nl_forward(w, d, srcs, recs)
    ref = O.nl_forward(g, c.vel, osrc, orec, w, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)


@pytest.mark.parametrize("nzi,nxi,shots,sub,every", [
    (64, 64, 1, 2, 0), (80, 48, 2, 2, 1), (112, 80, 3, 3, 7), (64, 112, 2, 2, 39), (176, 112, 5, 1, 20),
    (208, 240, 6, 2, 0), (208, 240, 6, 2, 11), (336, 272, 16, 2, 0), (336, 272, 16, 2, 13)])
def test_velocity_gradient(nzi, nxi, shots, sub, every):
    """Several steps per launch on 32 x 32, 64 x 32 and 64 x 64 tiles, one
    per launch where a receiver lies in the FAT ring, and the
    one-point-per-lane kernels with their imaging kernel."""
    A, c, ctx, g, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, sub, False, 40 // sub)
    m = c.wavelet[None, None, :].copy()
    dr = np.random.default_rng(6).standard_normal((shots, recs[0].nDev, c.nts)).astype(np.float32)
    if shots == 2:
        iz, ix = [2, 8], [9, 3]
        recs, orec = [A.Device.ints(iz, ix, c.nz, c.nx, c.nts)], [O.Device.ints(iz, ix, c.nz, c.nx, c.nts)]
        dr = dr[:, :2].copy()
    ref = O.nl_velocity_gradient(g, c.vel, osrc, orec, m, dr, "f")
    assert np.abs(ref).max() > 0
    for tile in (0, 3232):
        if tile:
            ctx.set_option("tileAdj", tile)
        grad = np.zeros((c.nx, c.nz), np.float32)
        ctx.nl_velocity_gradient(m, dr, grad, srcs, recs, checkpoint_every=every)
        np.testing.assert_array_equal(grad, ref)
