"""The advection kernel's launches by model and kind of order, in one batch:
every order, fluid tiles and tiles at walls, tiles clipped at the array's
edge, one and two tracers, with diffusion.  FP64 keeps the reference's
operations, so each instance equals the oracle bit for bit."""
import numpy as np
import pytest

from fluid2d_amd.batch import Batch
from tests.test_gpu_engine import init_fields, spec
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def test_orders_and_models_in_one_batch_vs_oracle():
    specs = [spec("euler", 96, 96, 1.0, 1.0, "closed", order=4),
             spec("euler", 256, 128, 2.0, 1.0, "perio", order=5),
             spec("euler", 128, 128, 1.0, 1.0, "disc", order=5, flux_splitting_method="minmax"),
             spec("euler", 192, 192, 1.0, 1.0, "closed", order=1),
             spec("boussinesq", 160, 96, 1.0, 0.6, "xchannel", order=3, diffusion=True, Kdiff=1e-4),
             spec("boussinesq", 256, 256, 1.0, 1.0, "closed", order=5, diffusion=True, Kdiff=1e-4),
             spec("boussinesq", 64, 32, 2.0, 1.0, "xchannel", order=6),
             spec("euler", 64, 64, 1.0, 1.0, "perio", order=2)]
    b = Batch(specs)
    fields = [init_fields(b, i, 40 + i) for i in range(len(specs))]
    for i, f in enumerate(fields):  # a moving start for every model
        if "buoyancy" in f:
            f["vorticity"] = f["vorticity"] * 0.5
            f["buoyancy"] = f["buoyancy"] + 0.1 * f["vorticity"]
            for k, v in f.items():
                b.set_field(i, k, v)
    b.set_psi_from_vorticity()
    orcs = []
    for i, f in enumerate(fields):
        p, g = b.params[i], b.grids[i]
        o = orc.OracleModel(p.modelname, g.nx, g.ny, g.Lx, g.Ly, geometry=g.geometry,
                            order=p.order, flux_splitting_method=p.flux_splitting_method,
                            diffusion=p.diffusion, Kdiff=p.Kdiff, gravity=p.gravity)
        for k, v in f.items():
            o.get(k)[...] = v
        o.set_psi_from_vorticity()
        ms = o.diagnostics()["maxspeed"]
        dt = 0.5 * min(g.dx, g.dy) / ms
        b.set_dt(dt, i)
        orcs.append((o, dt))
    b.step(3)
    for i, (o, dt) in enumerate(orcs):
        print("case rhs", specs[i], flush=True)
        o.run(3, dt)
        s = b.state(i)
        for k in range(s.shape[0]):
            assert np.array_equal(s[k], o.state[k]), "instance %d field %d" % (i, k)
