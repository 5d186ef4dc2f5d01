"""Node charge through the chunks of the last sort: FP64 against the global
deposit's, freshly sorted, with many particles outside their tile's window,
after a window shift with an unsorted tail, and the total charge."""
import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


def _rho(shape, ppc, sigma, deposit, steps, shift, precision="fp64"):
    rec, _ = oracle.synth_plasma(*shape, ppc, 0.02, sigma, 11)
    print(f"rho {shape} {ppc} {sigma} {deposit} {steps} {shift}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision=precision, deposit=deposit) as r:
        r.add_records(rec)
        pos = rec.copy()
        pos[:, 6:] = 0.01, 1.0
        r.add_records(pos[::3])
        r.init_boundaries()
        if steps:
            r.step(steps)
        if shift:
            r.moving_window()
            cells = np.array([(shape[0] - 3, j, k) for j in range(1, shape[1] - 2) for k in range(1, shape[2] - 2)], np.int32)
            r.fill_cells(0, cells, np.full(len(cells), 0.01), (1, 1, 1))
        return r.compute_rho(), r.particles(0)[0][:, 7].sum(), r.particles(1)[0][:, 7].sum()


@pytest.mark.parametrize("shape,ppc,sigma,steps,shift", [((8, 8, 8), 1, 0.1, 0, False), ((9, 17, 16), 3, 0.1, 1, False),
                                                         ((24, 17, 10), 9, 5.0, 9, False), ((33, 18, 19), 4, 0.1, 2, True),
                                                         ((33, 18, 19), 4, 5.0, 7, True)])
def test_tiled_rho_matches_global(shape, ppc, sigma, steps, shift):
    a, b = (_rho(shape, ppc, sigma, d, steps, shift) for d in ("tiled", "global"))
    # FP64 sums of some hundreds of terms in another order, positions alike to
    # 1e-12 after the steps; sums over the box of some 1e4
    assert np.abs(a[0] - b[0]).max() <= 1e-10 * np.abs(b[0]).max()
    for s in (0, 1):
        assert abs(a[0][..., s].sum() - a[1 + s]) <= 1e-10 * abs(a[1 + s])
    assert (a[0][..., 2] == 0).all()
