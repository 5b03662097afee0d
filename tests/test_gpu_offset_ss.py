"""The secondary sources and the imaging of the offset extension with four
z-points per lane (more than 11 offsets) give the float oracle's results bit
for bit: interior sizes that leave remainders of the 64 x 32 and 64 x 28 tiles,
grids narrower than the offsets' reach, offsets up to the kernels' bound and
beyond, odd shot counts (a workgroup takes two) and batches of samples, odd and
even, that do not divide the record."""
import numpy as np
import pytest

from cases import make_case
from oracle import oracle as O

pytestmark = pytest.mark.gpu
FAT = 5


@pytest.mark.parametrize("nzi,nxi,shots,nExt,batch", [
    (64, 64, 1, 21, 16), (80, 48, 3, 21, 7), (112, 80, 2, 13, 16), (48, 112, 5, 17, 1), (64, 48, 2, 23, 16)])
def test_extended_and_tomographic(nzi, nxi, shots, nExt, batch):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=nzi + nxi + nExt, nz=nzi + 2 * FAT, nx=nxi + 2 * FAT, nShot=shots, nts=30, sub=2, dts=0.002,
                  nExt=nExt, shot_dx=5)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=c.nts, dts=c.dts, sub=c.sub, zPadMinus=c.pad,
                         zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad, alphaCos=c.alpha, fMax=20.0, nExt=nExt,
                         extension=A.EXT_OFFSET))
    ctx.set_velocity(c.vel)
    ctx.set_option("extBatch", batch)
    srcs = [A.Device.grid(*a, c.nz, c.nx, c.nts) for _, a in c.src_args]
    recs = [A.Device.grid(*a, c.nz, c.nx, c.nts) for _, a in c.rec_args]
    os_, or_ = c.oracle_sources(), c.oracle_receivers()
    rng = np.random.default_rng(3)
    wav = c.wavelet[None, :].copy()
    m = rng.standard_normal((nExt, c.nx, c.nz)).astype(np.float32)
    d = np.zeros((shots, recs[0].nDev, c.nts), np.float32)
    ctx.bornext_forward(m, d, srcs, wav, recs)
    ref = O.bornext_forward(c.grid, c.vel, os_, [wav], or_, m, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    ctx.set_ext_reflectivity(m)
    ext = np.zeros_like(m)
    da = rng.standard_normal(d.shape).astype(np.float32)
    ctx.bornext_adjoint(ext, da, srcs, wav, recs)
    np.testing.assert_array_equal(ext, O.bornext_adjoint(c.grid, c.vel, os_, [wav], or_, da, "f"))
    dr = rng.standard_normal(d.shape).astype(np.float32)
    img = np.zeros((c.nx, c.nz), np.float32)
    ctx.tomo_adjoint(img, dr, srcs, wav, recs)
    np.testing.assert_array_equal(img, O.tomo_adjoint(c.grid, c.vel, os_, [wav], or_, dr, m))
