"""What the server books for a batch covers what the engine holds for it:
every request kind, one shot and several, on a model whose calls take several
fine steps per launch and on one whose Born forward keeps a ring."""
import numpy as np
import pytest

from cases import make_case
from acoustic_isotropic_operators_amd.serve import Request, Server

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nzi,nxi,sub,nExt,options", [
    (48, 64, 2, 5, {}), (112, 144, 2, 21, {}), (112, 144, 2, 21, {"extBatch": 4}), (80, 96, 4, 13, {}), (400, 640, 2, 3, {})])
def test_bookings_cover_the_engine(nzi, nxi, sub, nExt, options):
    c = make_case(seed=nzi, nz=nzi + 10, nx=nxi + 10, nShot=1, nts=40, sub=sub, dts=0.001 * sub, nExt=nExt)
    params = dict(nz=c.nz, nx=c.nx, dz=c.dz, dx=c.dx, nts=c.nts, dts=c.dts, sub=sub, zPadMinus=c.pad, zPadPlus=c.pad,
                  xPadMinus=c.pad, xPadPlus=c.pad, alphaCos=c.alpha, fMax=20.0)
    rng = np.random.default_rng(1)
    refl = rng.standard_normal((c.nx, c.nz)).astype(np.float32)
    for kind in ("nl_forward", "born_forward", "born_adjoint", "bornext_adjoint"):
        for n in (1, 5):
            srv = Server(max_models=1, nExt=nExt, options=options)
            srv.add_model("m", params, c.vel, c.rec_args[0][1], c.wavelet)
            nrec = srv.models["m"].rec[0].nDev
            for k in range(n):
                r = Request(kind, "m", (16, 15 + 3 * k))
                if kind == "born_forward":
                    r.payload, r.reflectivity_id = refl, 0
                elif kind != "nl_forward":
                    r.payload = rng.standard_normal((nrec, c.nts)).astype(np.float32)
                srv.submit(r)
            done = srv.step()
            assert len(done) == n and all(r.error is None for r in done)
            slot = srv.models["m"].slots[0]
            held = slot.ctx.info()["bytes_per_shot"] * n
            print(f"{kind}, {n} shots: booked {slot.reserved / 1e6:.2f} MB, held {held / 1e6:.2f} MB", flush=True)
            # a Born forward may book 1 GiB for the source slices of a short record
            assert held <= slot.reserved <= 1.5 * held + (32 << 20) + (kind == "born_forward") * (1 << 30)
            srv.models["m"].close()
