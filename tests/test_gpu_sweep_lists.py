"""The colours' schedule of the single-launch sweeps is made for solves that read it: natural-order solves leave it out."""
import pytest

from cfdsolutions_amd import cfd
from cfdsolutions_amd import mesh as cmesh

pytestmark = pytest.mark.gpu


def test_natural_order_solves_make_no_colour_lists():
    print("sweep lists", flush=True)
    ctx = cfd.Context(0)
    m = cmesh.bump_channel(24, 8, 8)
    p = cfd.make_params(mach=0.5, flux="roe", order=1)
    dm = cfd.DeviceMesh(ctx, m, p)
    dm.bc(p, 1)
    dm.residual(p)
    dm.delta_t(p, 1)
    dm.jacobian(p)
    held = []
    for precond in (cfd.PREC_ILU0, cfd.PREC_ILU0_MC, cfd.PREC_ILU0):
        dm.linsolve(precond=precond, krylov_m=5, max_restarts=0, rtol=1e-3)
        held.append(dm.device_bytes())
    assert held[1] >= held[0] + 2 * 4 * m.n_node and held[2] == held[1]
    dm.close()
    ctx.close()
