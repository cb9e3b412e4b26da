"""Fields on either side of the line between one plain copy of the records and the transfer by a kernel (64 KB: time
steps of 8,192 nodes, states of 1,024 nodes and ghosts in records of 8 values, residuals of 682 nodes in records of 12,
gradients of 409 in records of 20): each comes back as set, and one that is a part of its record leaves the rest alone."""
import types

import numpy as np
import pytest

from cfdsolutions_amd import cfd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [409, 410, 682, 683, 1023, 1024, 8192, 8193])
def test_fields_around_the_small_limit(n):
    print("fields", n, flush=True)
    ctx = cfd.Context(0)
    e = np.stack([np.arange(n - 1), np.arange(1, n)], 1).astype(np.int32)
    both = np.concatenate([e, e[:, ::-1]])
    both = both[np.lexsort((both[:, 1], both[:, 0]))]
    rng = np.random.default_rng(n)
    ia = np.concatenate([[0], np.cumsum(np.bincount(both[:, 0], minlength=n))]).astype(np.int32)
    m = types.SimpleNamespace(
        n_node=n, edge=e, edge_area=rng.standard_normal((n - 1, 3)), bedge=np.array([[0, n]], np.int32),
        bedge_area=np.ones((1, 3)), bedge_type=np.zeros(1, np.int32), bedge_tag=np.ones(1, np.int32),
        xyz=rng.standard_normal((n, 3)), vol=np.ones(n), n2n_ia=ia, n2n_ja=both[:, 1].astype(np.int32))
    dm = cfd.DeviceMesh(ctx, m, cfd.make_params())
    fields = [cfd.FIELD_DT, cfd.FIELD_GRAD, cfd.FIELD_PHI, cfd.FIELD_RES_CONV, cfd.FIELD_RES_DISS, cfd.FIELD_DT_ACC,
              cfd.FIELD_Q]
    want = {f: rng.standard_normal(dm._SHAPES[f](dm)) for f in fields}
    for f in fields:
        dm.set(f, want[f])
    for f in fields:
        assert np.array_equal(dm.get(f), want[f]), f
    dm.close()
    ctx.close()
