"""Read-backs at the edges of their blocks (qk_get_fields, qk_particle_count,
qk_get_particles): the values are those put in, exactly (FP64) or rounded to
FP32 once, whatever the number of blocks, workers and free slots."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


def region(shape, precision, **kw):
    return qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision=precision, deposit="global", **kw)


# 21845 nodes of three FP32 numbers fill a small slot, 174762 a large one
@pytest.mark.parametrize("shape", [(5, 5, 5), (29, 27, 28), (86, 32, 8), (141, 90, 91)])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_fields_come_back_as_set(shape, precision):
    rng = np.random.default_rng(sum(shape))
    E, B = rng.normal(size=shape + (3,)), rng.normal(size=shape + (3,))
    print(f"fields {shape} {precision}", flush=True)
    with region(shape, precision) as r:
        r.set_fields(E, B)
        got = r.get_fields()
    real = np.float32 if precision == "fp32" else np.float64
    np.testing.assert_array_equal(got[0], E.astype(real).astype(np.float64))
    np.testing.assert_array_equal(got[1], B.astype(real).astype(np.float64))
    assert not got[2].any() and not got[3].any()


@pytest.mark.parametrize("precision,ids", [("fp32", True), ("fp32", False), ("fp64", True)])
def test_live_particles_come_back_in_slot_order(precision, ids):
    shape = (40, 16, 16)
    real = np.float32 if precision == "fp32" else np.float64
    for n, shifts in ((1, 0), (1023, 0), (1024, 3), (1025, 39), (9000, 5), (600_001, 0), (600_001, 20)):
        rng = np.random.default_rng(n + shifts)
        cell = np.stack([rng.integers(1, m - 2, n) for m in shape], 1)
        off = rng.integers(0, 1 << 20, (n, 3)) / float(1 << 20)   # exact in FP32
        u, q = rng.normal(size=(n, 3)), rng.normal(size=n)
        pos = cell + off
        print(f"particles {n} {precision} ids {ids} shifts {shifts}", flush=True)
        with region(shape, precision, track_ids=ids) as r:
            r.add_particles(qa.ELECTRON, *pos.T, *u.T, q, ids=np.arange(n, dtype=np.int32))
            for _ in range(shifts):
                r.moving_window()
            live = cell[:, 0] >= shifts
            assert r.count(qa.ELECTRON) == live.sum()
            rec, got = r.particles(qa.ELECTRON)
        want = np.flatnonzero(live)
        np.testing.assert_array_equal(got, want if ids else np.zeros(len(want), int))
        np.testing.assert_array_equal(rec[:, :3], pos[live] - [shifts, 0, 0])
        uh = u[live].astype(real).astype(np.float64)
        np.testing.assert_array_equal(rec[:, 3:6], uh)
        np.testing.assert_allclose(rec[:, 6], np.sqrt(1 + (uh ** 2).sum(1)), rtol=4e-16)
        np.testing.assert_array_equal(rec[:, 7], q[live].astype(real).astype(np.float64))
        assert (rec[:, 8] == -1).all() and not rec[:, 9].any()


def test_short_output_buffer_is_refused():
    import ctypes as C
    with region((12, 12, 12), "fp32") as r:
        x = np.full(50, 5.5)
        r.add_particles(qa.ELECTRON, x, x, x, 0 * x, 0 * x, 0 * x, x)
        rec, ids, n = np.zeros((49, 10)), np.zeros(49, np.int32), C.c_int64(7)
        rc = qa.load_library().qk_get_particles(r._h, qa.ELECTRON, 49, rec.ctypes.data_as(C.POINTER(C.c_double)),
                                                ids.ctypes.data_as(C.POINTER(C.c_int32)), C.byref(n))
        assert rc == 2 and n.value == 0
