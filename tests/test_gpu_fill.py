"""qk_fill_cells at the edges of its groups of cells (64) and of the list that
goes through the pinned buffer (21845 cells), in fills that follow each other
with nothing waited for in between: every particle against the formula."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("counts,npic", [((1, 63, 2), (2, 2, 2)), ((64, 65, 127), (1, 2, 3)), ((21845, 21846, 5), (1, 1, 2))])
def test_fills_follow_each_other(counts, npic, precision):
    n = (40, 32, 32)
    i, j, k = np.meshgrid(np.arange(1, n[0] - 2), np.arange(1, n[1] - 2), np.arange(1, n[2] - 2), indexing="ij")
    cells = np.stack([i.ravel(), j.ravel(), k.ravel()], 1).astype(np.int32)
    npt = npic[0] * npic[1] * npic[2]
    want, first = [], 0
    print(f"fill {counts} {npic} {precision}", flush=True)
    with qa.Region(*n, DX, DX, DX, 0.5 * DX, precision=precision, track_ids=True) as r:
        for m, count in enumerate(counts):
            sel = cells[m * 7:m * 7 + count]
            dens = 0.01 + 1e-6 * np.arange(count)
            r.fill_cells(0, sel, dens, npic, 0.25, first)
            first += count * npt
            ip, jp, kp = (a.ravel() for a in np.meshgrid(*[np.arange(b) for b in npic], indexing="ij"))
            pos = [(sel[:, a, None] + 0.5 / npic[a] + p[None] / npic[a]).ravel() for a, p in enumerate((ip, jp, kp))]
            want.append(np.stack(pos + [np.repeat(-dens / npt, npt)], 1))
        rec, ids = r.particles(0)
    want = np.concatenate(want)
    assert sorted(ids) == list(range(len(want)))
    got = rec[np.argsort(ids)]
    tol = 1e-6 if precision == "fp32" else 1e-14   # one rounding of offset and charge
    assert np.abs(got[:, :3] - want[:, :3]).max() <= tol
    assert np.abs(got[:, 7] - want[:, 3]).max() <= tol * 0.05
    assert (got[:, 3] == 0.25).all() and (got[:, 4:6] == 0).all()
