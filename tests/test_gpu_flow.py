"""Single-launch sweeps whatever the GPU holds of a launch: one workgroup, a few, and more than it can hold at a time
(72x24x24 mesh: 2,800 workgroups of which 1,024 fit at most).  Chunks of rows go to the workgroups that run, so every
number gives the same bits and none waits for one that has not started."""
import numpy as np
import pytest

from cfdsolutions_amd import cfd
from cfdsolutions_amd import mesh as cmesh

pytestmark = pytest.mark.gpu

SOLVES = {
    "natural": dict(precond=cfd.PREC_ILU0),
    "colours": dict(precond=cfd.PREC_ILU0_MC),
    "gs": dict(solver=cfd.SOLVER_BLOCK_GS, sweeps=5),
    "lusgs": dict(solver=cfd.SOLVER_LUSGS, sweeps=2),
}


@pytest.fixture(scope="module")
def ctx():
    c = cfd.Context(0)
    yield c
    c.close()


def update(ctx, m, monkeypatch, blocks, mixed, kw):
    if blocks:
        monkeypatch.setenv("CFD_FLOW_BLOCKS", str(blocks))
    p = cfd.make_params(mach=0.5, alpha_deg=1.0, flux="roe", order=1, cfl_min=50.0)
    dm = cfd.DeviceMesh(ctx, m, p)
    monkeypatch.delenv("CFD_FLOW_BLOCKS", raising=False)
    dm.bc(p, 1)
    dm.residual(p)
    dm.delta_t(p, 1)
    dm.jacobian(p, mixed=mixed != 0)
    st = dm.linsolve(krylov_m=6, max_restarts=1, rtol=1e-12, mixed=mixed, **kw)
    x = dm.get(cfd.FIELD_X)
    dm.close()
    return st.iterations, st.final_res, x


@pytest.mark.parametrize("dims,blocks", [((12, 4, 4), 1), ((12, 4, 4), 3), ((72, 24, 24), 65536)],
                         ids=["one", "three", "more-than-fit"])
@pytest.mark.parametrize("solve,mixed", [("natural", 0), ("natural", 1), ("colours", 0), ("colours", 2), ("gs", 0),
                                         ("lusgs", 0)])
def test_any_number_of_workgroups(ctx, monkeypatch, dims, blocks, solve, mixed):
    print("flow", dims, blocks, solve, mixed, flush=True)
    m = cmesh.bump_channel(*dims)
    usual = update(ctx, m, monkeypatch, 0, mixed, SOLVES[solve])
    got = update(ctx, m, monkeypatch, blocks, mixed, SOLVES[solve])
    assert got[:2] == usual[:2] and np.array_equal(got[2], usual[2])
    assert np.all(np.isfinite(usual[2])) and np.any(usual[2] != 0.0)
