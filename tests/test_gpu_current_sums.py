"""The current of FP32 steps on grids whose tiles are cut into several chunks is
summed in FP64 and rounded once: in a step without fields, where every
particle's own numbers are the same in any order, J is the same in any order."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


# 27, 112 and 128 tiles in a part per CU, 150 and 432 in halves; two species
@pytest.mark.parametrize("shape,ppc,species", [((24, 23, 22), 9, 1), ((56, 32, 32), 8, 1), ((64, 32, 32), 8, 2),
                                               ((80, 39, 40), 8, 1), ((96, 48, 47), 10, 1)])
def test_sums_do_not_depend_on_their_order(shape, ppc, species):
    rng = np.random.default_rng(sum(shape))
    c = np.stack([x.ravel() for x in np.meshgrid(*[np.arange(1, n - 2) for n in shape], indexing="ij")], 1).repeat(ppc, 0)
    pos = c + rng.integers(0, 1 << 20, c.shape) / float(1 << 20)   # exact in FP32
    u = rng.normal(0, 0.05, c.shape).astype(np.float32)
    got = []
    for order in (np.arange(len(c)), np.arange(len(c)), rng.permutation(len(c))):
        print(f"current sums {shape} {ppc} {species}", flush=True)
        with qa.Region(*shape, DX, DX, DX, 0.5 * DX, solver="ndfx", pusher="vay", ion_cmr=(0.01,), track_ids=True) as r:
            for s in (qa.ELECTRON, qa.ION0)[:species]:
                r.add_particles(s, *pos[order].T, *u[order].T, np.full(len(c), -0.005 / ppc if s == 0 else 0.002 / ppc),
                                ids=order.astype(np.int32))
            r.init_boundaries()
            r.step(1)
            got.append((r.get_fields(), r.rows_by_id(qa.ELECTRON, len(c))[0]))
    assert np.abs(got[0][0][2]).max() > 0
    # an FP64 sum in another order differs by some 1e-15, and rounds to another
    # FP32 number where it lies that close to the middle of two (6e-8 apart): once
    # in 1e7 of the 1e5 to 7e5 numbers
    for fields, rows in got[1:]:
        assert (rows == got[0][1]).all()
        assert sum((a != b).sum() for a, b in zip(fields[:3], got[0][0][:3])) <= 3
