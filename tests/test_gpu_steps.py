"""The kernels that take several fine steps of a pass per launch give oracle's results bit for bit: interior sizes that leave remainders
of their 32 x 32, 64 x 32 and 64 x 64 tiles, step counts that are no multiple
of the steps per launch, sources and receivers on both sides of tile edges
and inside a neighbour's halo, sponges narrower and wider than a tile, more
receivers on a tile than it has threads, and shot counts on both sides of
the ones at which the tile changes."""
import numpy as np
import pytest

from cases import make_case
from oracle import oracle as O

pytestmark = pytest.mark.gpu
FAT = 5


def _setup(nzi, nxi, shots, sub, nts, pad, points):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=nzi * 7 + nxi, nz=nzi + 2 * FAT, nx=nxi + 2 * FAT, nShot=shots, nts=nts, sub=sub, pad=pad,
                  dts=0.001 * sub)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=c.nts, dts=c.dts, sub=c.sub, alphaCos=c.alpha,
                         fMax=20.0, zPadMinus=pad, zPadPlus=pad, xPadMinus=pad, xPadPlus=pad))
    ctx.set_velocity(c.vel)
    rng = np.random.default_rng(9)
    # sources next to tile edges, receivers as asked for
    at = [(FAT + min(nzi - 1, 31 + s % 3), FAT + (s * 31 + 30) % nxi) for s in range(shots)]
    if points == "all":
        iz, ix = (v.ravel().tolist() for v in np.mgrid[FAT:FAT + nzi, FAT:FAT + nxi])
    else:
        iz = [FAT, FAT + nzi - 1] + [FAT + (17 * k) % nzi for k in range(points)]
        ix = [FAT, FAT + nxi - 1] + [FAT + (5 * k) % nxi for k in range(points)]
        iz, ix = (list(v) for v in zip(*sorted(set(zip(iz, ix)))))
    dims = (c.nz, c.nx, c.nts)
    srcs = [A.Device.ints([z], [x], *dims) for z, x in at]
    osrc = [O.Device.ints([z], [x], *dims) for z, x in at]
    recs, orec = [A.Device.ints(iz, ix, *dims)], [O.Device.ints(iz, ix, *dims)]
    return c, ctx, rng, srcs, recs, osrc, orec


def _check(nzi, nxi, shots, sub, nts, pad, points):
    c, ctx, rng, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, sub, nts, pad, points)
    g = c.grid
    w = rng.standard_normal((shots, 1, nts)).astype(np.float32)
    d = np.zeros((shots, recs[0].nDev, nts), np.float32)
    ctx.nl_forward(w, d, srcs, recs)
    ref = O.nl_forward(g, c.vel, osrc, orec, w, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    dr = rng.standard_normal(d.shape).astype(np.float32)
    m = np.zeros((shots, 1, nts), np.float32)
    ctx.nl_adjoint(m, dr, srcs, recs)
    np.testing.assert_array_equal(m, O.nl_adjoint(g, c.vel, osrc, orec, dr, shots, "f"))


@pytest.mark.parametrize("nzi,nxi,shots,sub,nts,pad", [
    (32, 32, 1, 2, 2, 10),         # one tile, two steps
    (48, 80, 1, 4, 12, 10),        # remainders of 16
    (64, 96, 2, 3, 18, 4),         # 51 steps: a last launch of 3
    (112, 80, 1, 1, 40, 40),       # sponge wider than a tile, 39 steps
    (208, 240, 6, 2, 20, 10),      # 64 x 32 tiles, 38 steps: a last launch of 2
    (208, 240, 14, 2, 21, 10),     # 64 x 64 tiles, 40 steps: a last launch of 1
    (208, 256, 26, 4, 8, 50),      # 416 workgroups, two rounds
    (272, 304, 24, 2, 12, 10),     # one step per launch again
])
def test_nonlinear_passes(nzi, nxi, shots, sub, nts, pad):
    _check(nzi, nxi, shots, sub, nts, pad, 37)


def test_more_receivers_than_threads():
    _check(64, 64, 1, 2, 9, 10, "all")
    _check(64, 64, 60, 2, 5, 10, "all")


@pytest.mark.parametrize("nzi,nxi,shots,sub,nts,pad", [
    (32, 32, 1, 2, 2, 10),
    (48, 80, 1, 4, 12, 10),
    (64, 96, 2, 3, 18, 4),
    (112, 80, 1, 1, 40, 40),
    (208, 240, 6, 2, 20, 10),
    (208, 240, 6, 3, 14, 10),
    (208, 240, 14, 2, 21, 10),
    (208, 240, 14, 4, 11, 10),
    (208, 256, 26, 2, 14, 50),
    (272, 304, 24, 2, 12, 10),
])
def test_born_passes(nzi, nxi, shots, sub, nts, pad):
    c, ctx, rng, srcs, recs, osrc, orec = _setup(nzi, nxi, shots, sub, nts, pad, 37)
    g = c.grid
    wav = rng.standard_normal((1, nts)).astype(np.float32)
    m = rng.standard_normal((c.nx, c.nz)).astype(np.float32)
    d = np.zeros((shots, recs[0].nDev, nts), np.float32)
    ctx.born_forward(m, d, srcs, wav, recs)
    ref = O.born_forward(g, c.vel, osrc, [wav], orec, m, "f")
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(d, ref)
    dr = rng.standard_normal(d.shape).astype(np.float32)
    img = np.zeros((c.nx, c.nz), np.float32)
    ctx.born_adjoint(img, dr, srcs, wav, recs)
    np.testing.assert_array_equal(img, O.born_adjoint(g, c.vel, osrc, [wav], orec, dr, "f"))


@pytest.mark.parametrize("nzi,nxi,shots", [(640, 832, 10), (640, 832, 21), (640, 832, 1), (2064, 2576, 2)])
def test_gradient_batches(nzi, nxi, shots):
    """The velocity gradient's own split into batches gives the bits of one
    batch of all shots: one batch, several of equal and of unequal sizes, and
    a batch for each shot."""
    c, ctx, rng, srcs, recs, _, _ = _setup(nzi, nxi, shots, 2, 12, 20, 9)
    m = rng.standard_normal((1, 1, c.nts)).astype(np.float32)
    d = rng.standard_normal((shots, recs[0].nDev, c.nts)).astype(np.float32)
    one, split = (np.zeros(c.vel.shape, np.float32) for _ in range(2))
    ctx.nl_velocity_gradient(m, d, split, srcs, recs)
    ctx.set_option("batchAdj", shots)
    ctx.nl_velocity_gradient(m, d, one, srcs, recs)
    assert np.any(one) and np.array_equal(one, split)


@pytest.mark.parametrize("nts", [2, 3, 17, 60])
def test_gradient_first_and_later_calls(nts):
    """A context's first velocity gradient, in short segments, and the later
    ones, in as few as fit, give the bits of one segment per step."""
    c, ctx, rng, srcs, recs, _, _ = _setup(48, 80, 2, 2, nts, 20, 9)
    m = rng.standard_normal((1, 1, c.nts)).astype(np.float32)
    d = rng.standard_normal((2, recs[0].nDev, c.nts)).astype(np.float32)
    first, second, third, ref = (np.zeros(c.vel.shape, np.float32) for _ in range(4))
    for g, every in ((first, 0), (second, 0), (ref, 1), (third, 0)):
        ctx.nl_velocity_gradient(m, d, g, srcs, recs, checkpoint_every=every)
    for g in (first, second, third):
        assert np.array_equal(g, ref)
    assert nts < 60 or np.any(ref)      # the waves have met
