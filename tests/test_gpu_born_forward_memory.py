"""The Born forward with two fine steps per sample keeps three coarse slices
of the source field where a record's slices would take too much memory, and
all of them only for short records of few points; either form gives the same
bits."""
import numpy as np
import pytest

from cases import make_case

pytestmark = pytest.mark.gpu


def _call(nzi, nxi, shots, nts, **options):
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=8, nz=nzi + 10, nx=nxi + 10, nShot=shots, nts=nts, sub=2, dts=0.002, shot_dx=3)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=nts, dts=c.dts, sub=2, zPadMinus=c.pad,
                         zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad, alphaCos=c.alpha, fMax=20.0))
    ctx.set_velocity(c.vel)
    for k, v in options.items():
        ctx.set_option(k, v)
    srcs = [A.Device.grid(*a, c.nz, c.nx, nts) for _, a in c.src_args]
    recs = [A.Device.ints([20], [30], c.nz, c.nx, nts)]
    m = np.random.default_rng(9).standard_normal((c.nx, c.nz)).astype(np.float32)
    d = np.zeros((shots, 1, nts), np.float32)
    ctx.born_forward(m, d, srcs, c.wavelet[None, :].copy(), recs)
    info = ctx.info()
    traces = 4 * (nts * recs[0].nReg + ((nts - 1) * 2 + 1) * srcs[0].nReg)
    return d, (info["bytes_per_shot"] - traces) / (4.0 * c.nz * c.nx), info["batch"]


def test_a_long_record_keeps_the_ring():
    nts = 40000                                                      # 1.4 GB of slices of 64 x 112 points
    d, slices, _ = _call(64, 112, 1, nts)
    assert slices < 10
    ref, _, _ = _call(64, 112, 1, nts, tileFwd=3216)                 # one step per launch, lockstep
    assert np.any(ref) and np.array_equal(d, ref)


def test_a_short_record_keeps_every_slice():
    d, slices, _ = _call(64, 112, 1, 200)
    assert 200 <= slices < 210
    ref, slices, _ = _call(64, 112, 1, 200, tileFwd=3216)
    assert slices < 10 and np.any(ref) and np.array_equal(d, ref)


def test_the_form_follows_the_shots_of_a_launch():
    d, slices, batch = _call(208, 240, 12, 30, batchFwd=4)           # 4 of 32 tiles of 64 x 32 each run at once
    assert batch == 4 and 30 <= slices < 40
    ref, slices, _ = _call(208, 240, 12, 30)                         # 12 do not
    assert slices < 10 and np.any(ref) and np.array_equal(d, ref)
