"""Rows of a mesh's multicolour pattern that are sorted by a whole wavefront: of one block more than one lane's limit, of
a power of two, one more, and thousands.  Seen through the multicolour ILU(0), whose result on them equals the oracle's
on the system in the colours' order (rounding: 20 eps a block of the longest row)."""
import numpy as np
import pytest

from cfdsolutions_amd import cfd
from oracle import oracle as orc

from test_gpu_ilu_rows import direction, late_rows, multicolour

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cfd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("blocks", [32, 33, 64, 65, 3001])
def test_multicolour_pattern_of_long_rows(ctx, blocks):
    print("hub row", blocks, flush=True)
    m = late_rows(2 * blocks, 3, blocks - 1)
    dm = cfd.DeviceMesh(ctx, m, cfd.make_params())
    ia, ja, iau = dm.bsr_structure()
    assert np.diff(ia).max() == blocks
    rng = np.random.default_rng(blocks)
    a = rng.uniform(-1.0, 1.0, (ja.size, 25))
    a[iau] += (np.diff(ia)[:, None] * 3.0 + 2.0) * np.eye(5).ravel()
    b = rng.uniform(-1.0, 1.0, (m.n_node, 5))
    dm.jacobian_set(a, b)
    dm.linsolve(precond=cfd.PREC_ILU0_MC, krylov_m=1, max_restarts=0, rtol=1e-30)
    x = dm.get(cfd.FIELD_X).reshape(-1, 5)
    dm.close()
    perm, _, ia, ja, iau, a, b = multicolour(ia, ja, iau, a, b)
    lu, dinv, rc = orc.ilu0(ia, ja, iau, a)
    assert rc == 0
    z, x = direction(orc.ilu0_apply(ia, ja, iau, lu, dinv, b).reshape(-1, 5)), direction(x[perm])
    assert min(np.linalg.norm(x - z), np.linalg.norm(x + z)) <= 20 * blocks * np.finfo(float).eps
