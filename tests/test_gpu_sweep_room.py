"""Gauss-Seidel sweeps with little device memory left: up to 32 sweeps share a launch, each with a version of x, where
there is room, and fewer, down to one, where there is not; x and the RMS are the same.  The shortage is forced from the
host: CFD_MESH_BYTES_MAX makes allocations of a mesh past that many bytes fail as the device's own would."""
import numpy as np
import pytest

from cfdsolutions_amd import cfd
from cfdsolutions_amd import mesh as cmesh

pytestmark = pytest.mark.gpu


def solve(ctx, m, sweeps, room=None, monkeypatch=None):
    p = cfd.make_params(mach=0.5, alpha_deg=1.0, flux="roe", order=1, cfl_min=5.0)
    if room is not None:
        monkeypatch.setenv("CFD_MESH_BYTES_MAX", str(room))
    dm = cfd.DeviceMesh(ctx, m, p)
    monkeypatch.delenv("CFD_MESH_BYTES_MAX", raising=False)
    dm.bc(p, 1)
    dm.residual(p)
    dm.delta_t(p, 1)
    dm.jacobian(p)
    before = dm.device_bytes()
    try:
        for _ in range(2):  # a second solve does not try again for what there is no room for
            st = dm.linsolve(solver=cfd.SOLVER_BLOCK_GS, sweeps=sweeps)
        return before, dm.device_bytes(), (st.iterations, st.final_res), dm.get(cfd.FIELD_X)
    finally:
        dm.close()


@pytest.mark.parametrize("versions", [0, 1, 2, 7, 31])
def test_fewer_sweeps_a_launch_where_memory_is_short(monkeypatch, versions):
    print("sweeps with room for", versions, flush=True)
    ctx = cfd.Context(0)
    m = cmesh.bump_channel(36, 12, 12)
    one = 48 * m.n_node
    before, after, stats, x = solve(ctx, m, 33, monkeypatch=monkeypatch)
    assert after >= before + 32 * one + 200 * m.n_node
    room = before + 200 * m.n_node + 64 + versions * one  # the factors of the diagonal blocks, and so many versions
    if versions == 0:
        with pytest.raises(cfd.CfdError) as e:
            solve(ctx, m, 33, room, monkeypatch)
        assert e.value.code == cfd.E_OOM
    else:  # the schedule of sweeps that share a launch comes first or not at all
        _, held, stats2, x2 = solve(ctx, m, 33, room, monkeypatch)
        assert held <= room
        assert stats2 == stats and np.array_equal(x2, x)
    ctx.close()
