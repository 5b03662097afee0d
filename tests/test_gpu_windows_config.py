"""A batch of windows reports the configuration that its calls run, and
setting what it reports changes nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("windows,tx,spl", [(8, 32, 4), (2, 16, 0)])
def test_reported_configuration_is_the_one_that_runs(windows, tx, spl):
    from acoustic_isotropic_operators_amd import _capi as A
    nz, nx, nts = 778, 1002, 40                                      # 24 x 31 tiles of 32 x 32 each
    b = A.Batch(dict(nz=nz, nx=nx, dz=10.0, dx=10.0, nts=nts, dts=0.002, sub=2, zPadMinus=10, zPadPlus=10,
                     xPadMinus=10, xPadPlus=10, alphaCos=0.95, fMax=20.0))
    vel = np.full((nx, nz), 2000.0, np.float32)
    b.set_windows([vel] * windows, [A.Device.grid(1, 300, 1, 1, 40 * k + 20, 1, nz, nx, nts) for k in range(windows)],
                  [A.Device.grid(1, 305, 1, 30, 20, 10, nz, nx, nts)] * windows)
    cfg, info = b.config(), b.info()
    assert (cfg["tz"], cfg["tx"], cfg["windows_per_launch"]) == (32, tx, spl)
    w = np.zeros((1, nts), np.float32)
    w[0, :8] = 1.0
    before = [np.zeros((30, nts), np.float32) for _ in range(windows)]
    b.nl_forward([w], before)
    b.set_config(**cfg)
    assert b.config() == cfg and b.info()["launch_groups"] == info["launch_groups"]
    after = [np.zeros((30, nts), np.float32) for _ in range(windows)]
    b.nl_forward([w], after)
    assert np.any(before[0]) and all(np.array_equal(x, y) for x, y in zip(before, after))
