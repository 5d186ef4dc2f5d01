"""Read-backs on both sides of the sizes from which helper threads share them,
and again in the same context, which then shares smaller ones too: fields,
node charges, records and rows by id are the same numbers either way."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


# 28 MiB are 611669.3 nodes of four FP32 fields
@pytest.mark.parametrize("shape,precision", [((50, 111, 110), "fp32"), ((85, 85, 85), "fp32"), ((50, 53, 115), "fp64"),
                                             ((67, 68, 68), "fp64")])
def test_fields(shape, precision):
    rng = np.random.default_rng(sum(shape))
    E, B = rng.normal(size=(2,) + shape + (3,)).astype(np.float32 if precision == "fp32" else np.float64)
    print(f"read-back sizes, fields {shape} {precision}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision=precision) as r:
        r.set_fields(E, B)
        for _ in range(2):
            got = r.get_fields()
            assert (got[0] == E).all() and (got[1] == B).all() and not got[2].any() and not got[3].any()


# 12 MiB are 349525.3 records of 36 bytes, 40 MiB 748982.9 rows by id
@pytest.mark.parametrize("n", [349525, 349526, 748982, 748983])
def test_records_and_rows(n):
    shape = (40, 20, 24)
    rng = np.random.default_rng(n)
    cell = np.stack([rng.integers(1, m - 2, n) for m in shape], 1)
    pos = cell + rng.integers(0, 1 << 20, (n, 3)) / float(1 << 20)   # exact in FP32
    u = rng.normal(size=(n, 3)).astype(np.float32)
    print(f"read-back sizes, records {n}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, track_ids=True) as r:
        r.add_particles(qa.ELECTRON, *pos.T, *u.T, np.full(n, -0.5), ids=np.arange(n, dtype=np.int32))
        for _ in range(2):
            rec, ids = r.particles(qa.ELECTRON)
            assert (ids == np.arange(n)).all() and (rec[:, :3] == pos).all() and (rec[:, 3:6] == u).all()
            rows, live = r.rows_by_id(qa.ELECTRON, n)
            assert live.all() and (rows[:, :6] == rec[:, :6]).all() and (rows[:, 6] == -0.5).all()


# 40 MiB are 1747626.7 nodes of three charges
@pytest.mark.parametrize("shape", [(120, 120, 121), (121, 121, 121)])
def test_node_charges(shape):
    print(f"read-back sizes, charges {shape}", flush=True)
    n = 5000
    rng = np.random.default_rng(1)
    cell = np.stack([rng.integers(1, m - 2, n) for m in shape], 1)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX) as r:
        r.add_particles(qa.ELECTRON, *cell.T.astype(float), *np.zeros((3, n)), np.full(n, -0.25))   # on the nodes
        want = np.zeros(shape + (3,))
        np.add.at(want[..., 0], tuple(cell.T), -0.25)
        for _ in range(2):
            assert (r.compute_rho() == want).all()
