"""ILU(0) rows that do not fit the factorisation's registers and LDS, in both precisions: rows of up to 60 blocks, in
levels of a few rows, of some thousand (one row to a wavefront) and of more (12 rows to a wavefront), a row of hundreds,
and the same in FP32 from an assembled Jacobian.

One FGMRES step gives x = y M^-1 b, whose direction is the oracle's preconditioned b.  In FP64 it differs by rounding
alone: of `blocks` blocks in the longest row each entry takes 5 `blocks` products twice over (factors, sweeps), and the
rows' dominance keeps errors from growing, so 20 blocks eps bounds the relative error; in FP32 the same with its eps.
"""
import types

import numpy as np
import pytest

from cfdsolutions_amd import cfd
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cfd.Context(0)
    yield c
    c.close()


def late_rows(early, late, most, seed=9):
    """A chain of `early` nodes, then `late` nodes that only know 10..most of the chain's (all of one colour, their
    neighbours all before them), the last of them exactly `most`."""
    rng = np.random.default_rng(seed)
    k = rng.integers(10, most + 1, late)
    k[-1] = most
    row = np.repeat(np.arange(late), k)
    at = rng.integers(0, early, row.size)
    e = np.unique(np.stack([at, early + row], 1), axis=0)
    missing = np.setdiff1d(np.arange(0, 2 * most), e[e[:, 1] == early + late - 1, 0])[:most]
    have = (e[:, 1] == early + late - 1).sum()
    e = np.concatenate([np.stack([np.arange(early - 1), np.arange(1, early)], 1), e,
                        np.stack([missing[:most - have], np.full(most - have, early + late - 1)], 1)]).astype(np.int32)
    n = early + late
    both = np.concatenate([e, e[:, ::-1]])
    both = both[np.lexsort((both[:, 1], both[:, 0]))]
    ia = np.concatenate([[0], np.cumsum(np.bincount(both[:, 0], minlength=n))]).astype(np.int32)
    return types.SimpleNamespace(
        n_node=n, edge=e, edge_area=0.1 * rng.standard_normal((len(e), 3)), bedge=np.array([[0, n]], np.int32),
        bedge_area=np.ones((1, 3)), bedge_type=np.zeros(1, np.int32), bedge_tag=np.ones(1, np.int32),
        xyz=rng.standard_normal((n, 3)), vol=np.ones(n), n2n_ia=ia, n2n_ja=both[:, 1].astype(np.int32))


def multicolour(ia, ja, iau, a, b):
    """The system with its rows in the order of a greedy colouring (in row order), ties by row."""
    n = ia.size - 1
    colour = np.full(n, -1)
    for i in range(n):
        used = set(colour[ja[ia[i]:ia[i + 1]]].tolist())
        c = 0
        while c in used:
            c += 1
        colour[i] = c
    perm = np.argsort(colour, kind="stable")
    inv = np.empty(n, np.int64)
    inv[perm] = np.arange(n)
    row = inv[np.repeat(np.arange(n), np.diff(ia))]
    at = np.lexsort((inv[ja], row))
    pia = np.concatenate([[0], np.cumsum(np.diff(ia)[perm])]).astype(np.int32)
    pja = inv[ja][at].astype(np.int32)
    piau = np.flatnonzero(pja == row[at]).astype(np.int32)
    return perm, np.diff(np.append(np.flatnonzero(np.diff(colour[perm], prepend=-1)), n)), pia, pja, piau, a[at], b[perm]


# early, late nodes, longest late row's neighbours; narrow: up to 4096 rows a level, or 32,768 in FP64 where one row in 16
# is long; wide: above (FP64: late rows fewer than one in 16)
CASES = [(200, 40, 60), (400, 30, 390), (6000, 3000, 24), (30000, 9000, 60), (190000, 10000, 60)]


def direction(x):
    return x / np.linalg.norm(x)


@pytest.mark.parametrize("precond", [cfd.PREC_ILU0, cfd.PREC_ILU0_MC], ids=["natural", "colours"])
@pytest.mark.parametrize("mixed", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("early,late,most", CASES)
def test_long_rows_equal_oracle(ctx, early, late, most, mixed, precond):
    print("long rows", early, late, most, mixed, precond, flush=True)
    if precond == cfd.PREC_ILU0 and early > 30000:
        pytest.skip("a natural-order chain of that length is only slow")
    m = late_rows(early, late, most)
    p = cfd.make_params(mach=0.3, flux="roe", order=1, cfl_min=0.1, cfl_max=0.1)
    dm = cfd.DeviceMesh(ctx, m, p)
    ia, ja, iau = dm.bsr_structure()
    n = m.n_node
    rng = np.random.default_rng(n)
    if mixed:
        q = dm.get(cfd.FIELD_Q)
        q *= 1.0 + 0.05 * rng.uniform(-1.0, 1.0, q.shape)
        dm.set(cfd.FIELD_Q, q)
        dm.residual(p)
        dm.delta_t(p, 1)
        dm.jacobian(p, mixed=True)
        a, b = dm.jacobian_get()
        a = a.reshape(-1, 25)
        b = b.reshape(n, 5)
    else:
        a = rng.uniform(-1.0, 1.0, (ja.size, 25))
        a[iau] += (np.diff(ia)[:, None] * 3.0 + 2.0) * np.eye(5).ravel()
        b = rng.uniform(-1.0, 1.0, (n, 5))
        dm.jacobian_set(a, b)
    dm.linsolve(precond=precond, krylov_m=1, max_restarts=0, rtol=1e-30, mixed=mixed)
    x = dm.get(cfd.FIELD_X).reshape(n, 5)
    dm.close()
    blocks = np.diff(ia).max()
    assert blocks == most + 1
    if precond == cfd.PREC_ILU0_MC:
        perm, widths, ia, ja, iau, a, b = multicolour(ia, ja, iau, a, b)
        assert late in widths  # the late rows are one level
        x = x[perm]
    lu, dinv, rc = orc.ilu0(ia, ja, iau, a)
    assert rc == 0
    z = direction(orc.ilu0_apply(ia, ja, iau, lu, dinv, b).reshape(-1, 5))
    x = direction(x)
    if np.vdot(x, z) < 0:
        x = -x
    tol = 20 * blocks * np.finfo(np.float32 if mixed else np.float64).eps
    assert np.linalg.norm(x - z) <= tol
    if not mixed:  # the updates decide: with A's own diagonal in the late rows the direction is another
        d = np.linalg.inv(a[iau[-late:]].reshape(-1, 5, 5)).reshape(-1, 25)
        other = direction(orc.ilu0_apply(ia, ja, iau, lu, np.concatenate([dinv[:-late], d]), b).reshape(-1, 5))
        assert np.linalg.norm(other - z) > 20 * tol
