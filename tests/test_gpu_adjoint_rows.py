"""Rows by id and rows by slot give one gradient: with particles deleted on
the way, in one block of rows and in two, in both deposits; and ids that are
no permutation are refused."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi
SHAPE = (20, 18, 17)


def _run(n, deposit, by_id, ids=None, steps=2):
    rng = np.random.default_rng(8)
    lo, hi = np.array([1.0, 1.0, 1.0]), np.array(SHAPE) - 2.0
    pos = lo + (hi - lo) * rng.random((n, 3))
    u = rng.normal(0, 1.0, (n, 3))
    E, B = rng.uniform(-0.1, 0.1, SHAPE + (3,)), rng.uniform(-0.1, 0.1, SHAPE + (3,))
    lam = rng.normal(0, 1, (n, 7))
    lE, lB = rng.normal(0, 1, SHAPE + (3,)), rng.normal(0, 1, SHAPE + (3,))
    given = ids is not None
    ids = ids if given else np.random.default_rng(9).permutation(n).astype(np.int32)
    print(f"adjoint rows {n} {deposit} {by_id}", flush=True)
    with qa.Region(*SHAPE, DX, DX, DX, 0.5 * DX, precision="fp64", deposit=deposit, track_ids=True) as r:
        r.set_fields(E, B)
        r.add_particles(0, *pos.T, *u.T, np.full(n, -0.01 * len(pos[:100]) / n), ids=ids)
        r.init_boundaries()
        r.tape_begin(2)
        r.step(steps)
        rec, left = r.particles(0)
        if given:
            return r.adjoint_by_id(lE, lB, {0: lam})
        rows, live = r.rows_by_id(0, n)
        assert (np.flatnonzero(live) == np.sort(left)).all() and (rows[~live] == 0).all()
        assert (rows[left] == rec[:, [0, 1, 2, 3, 4, 5, 7]]).all()
        if by_id:
            gE, gB, gp = r.adjoint_by_id(lE, lB, {0: lam})
            return gE, gB, gp[0], len(left)
        order, alive = r.tape_ids(0), np.zeros(n, bool)
        alive[left] = True
        gE, gB, gp = r.adjoint(lE, lB, {0: (lam * alive[:, None])[order]})
        g = np.zeros((n, 7))
        g[order] = gp[0]
        return gE, gB, g, len(left)


# 64 MiB hold 1198372 rows
@pytest.mark.parametrize("n,deposit", [(1, "tiled"), (4097, "tiled"), (4097, "global"), (1198373, "tiled")])
def test_rows_by_id_are_rows_by_slot(n, deposit):
    a, b = _run(n, deposit, True), _run(n, deposit, False)
    assert a[3] == b[3] and (a[3] < n or n == 1)
    for x, y in zip(a[:3], b[:3]):
        # FP64 sums in another order: some 1e3 terms per node
        assert np.abs(x - y).max() <= 1e-11 * np.abs(y).max()


def test_ids_outside_the_rows_are_refused():
    with qa.Region(*SHAPE, DX, DX, DX, 0.5 * DX, track_ids=True) as r:
        r.add_particles(0, *[np.full(3, 5.5)] * 3, *[np.zeros(3)] * 3, np.full(3, -0.01), ids=np.array([0, 3, 1], np.int32))
        with pytest.raises(qa.QuillError):
            r.rows_by_id(0, 3)
        assert (r.rows_by_id(0, 4)[1] == [True, True, False, True]).all()


def test_other_ids_are_refused():
    for ids in (np.arange(1, 11), np.array([0, 1, 2, 3, 4, 5, 6, 7, 8, 8])):
        with pytest.raises(qa.QuillError):
            _run(10, "global", True, ids.astype(np.int32))
