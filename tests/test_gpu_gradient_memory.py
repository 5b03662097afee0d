"""The velocity gradient's device memory: a context's later gradients take no
more than its first one, which holds the slices of segments of 2 sqrt(T)
steps and their checkpoints, and every call gives the same bits."""
import numpy as np
import pytest

from cases import make_case

pytestmark = pytest.mark.gpu


def test_later_gradients_take_no_more_memory_than_the_first():
    import torch
    from acoustic_isotropic_operators_amd import _capi as A
    c = make_case(seed=5, nz=218, nx=250, nShot=4, nts=400, sub=2, dts=0.002)
    ctx = A.Context(dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=c.nts, dts=c.dts, sub=c.sub, zPadMinus=c.pad,
                         zPadPlus=c.pad, xPadMinus=c.pad, xPadPlus=c.pad, alphaCos=c.alpha, fMax=20.0))
    ctx.set_velocity(c.vel)
    srcs = [A.Device.grid(*a, c.nz, c.nx, c.nts) for _, a in c.src_args]
    recs = [A.Device.grid(*a, c.nz, c.nx, c.nts) for _, a in c.rec_args]
    m = c.wavelet[None, None, :].copy()
    d = np.random.default_rng(6).standard_normal((c.nShot, recs[0].nDev, c.nts)).astype(np.float32)
    free, grads = [torch.cuda.mem_get_info()[0]], []
    for _ in range(3):
        g = np.zeros((c.nx, c.nz), np.float32)
        ctx.nl_velocity_gradient(m, d, g, srcs, recs)
        grads.append(g)
        free.append(torch.cuda.mem_get_info()[0])
    print("free memory before and after each call, MB:", [f >> 20 for f in free], flush=True)
    assert np.any(grads[0]) and np.array_equal(grads[0], grads[1]) and np.array_equal(grads[0], grads[2])
    assert free[2] == free[1] and free[3] == free[1]
    # 3 sqrt(T) slices per shot of W and checkpoints, 9 more of the fields and
    # the image, and the traces; the allocator rounds each buffer up
    T = (c.nts - 1) * c.sub
    slices = c.nShot * c.nz * c.nx * 4 * (3 * int(np.ceil(np.sqrt(T))) + 9 + 2)
    assert free[0] - free[1] < slices + (64 << 20)
