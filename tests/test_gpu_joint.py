"""The joint tiled push (one workgroup takes every species' particles of a
tile): FP64 against the global deposit on the same inputs, with two to four
species of unlike numbers, one of them on few tiles, tiles in parts, and a
species sorted apart from the others across a window shift."""
import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


def _species(shape, ppc, seed):
    """Electrons everywhere, positrons in a corner, two ion species."""
    rec = []
    for m, (p, cmr) in enumerate(zip(ppc, (-1.0, 1.0, 1 / 1836, 1 / 3672))):
        if p == 0:
            continue
        r, _ = oracle.synth_plasma(*shape, p, 0.02, 0.3, seed + m)
        r[:, 6] = np.abs(r[:, 6]) * np.sign(cmr)
        r[:, 7] = cmr
        if cmr == 1.0:
            r = r[(r[:, 0] < 9) & (r[:, 1] < 9)]
        rec.append(r)
    return np.concatenate(rec)


def _run(shape, ppc, deposit, shift_at=None, precision="fp64"):
    rng = np.random.default_rng(2)
    E, B = rng.uniform(-0.1, 0.1, shape + (3,)), rng.uniform(-0.1, 0.1, shape + (3,))
    print(f"joint {shape} {ppc} {deposit} {shift_at}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision=precision, deposit=deposit, sort_every=2,
                   ion_cmr=(1 / 1836, 1 / 3672)) as r:
        r.set_fields(E, B)
        r.add_records(_species(shape, ppc, 11))
        r.init_boundaries()
        d = []
        for step in range(5):
            if step == shift_at:
                r.moving_window()
                # positrons enough for a sort of theirs alone
                cells = np.array([(i, j, k) for i in range(1, 6) for j in range(1, 6) for k in range(1, 6)], np.int32)
                r.fill_cells(qa.POSITRON, cells, np.full(len(cells), 0.01), (2, 2, 2))
            d += r.step(1, diag=True)
        return r.get_fields(), d


@pytest.mark.parametrize("shape,ppc", [((8, 8, 8), (1, 1, 0, 0)), ((17, 9, 10), (40, 9, 3, 1)),
                                       ((33, 34, 35), (3, 2, 3, 0)), ((12, 12, 12), (150, 0, 150, 0)),
                                       ((66, 32, 31), (4, 0, 4, 0))])
def test_joint_matches_global_deposit(shape, ppc):
    (fg, dg), (ft, dt) = _run(shape, ppc, "global"), _run(shape, ppc, "tiled")
    for a, b in zip(ft, fg):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    for a, b in zip(dt, dg):
        assert a["n_e"] == b["n_e"] and a["n_p"] == b["n_p"] and a["n_ion"] == b["n_ion"]
        for k in ("energy_e", "energy_p", "energy_ion"):
            assert abs(a[k] - b[k]) <= 1e-12 * abs(b[k])


def test_species_sorted_apart_across_a_shift():
    (fg, dg), (ft, dt) = (_run((33, 18, 19), (3, 2, 3, 0), d, shift_at=3) for d in ("global", "tiled"))
    for a, b in zip(ft, fg):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    assert dt[-1]["n_p"] == dg[-1]["n_p"] and dt[-1]["n_e"] == dg[-1]["n_e"]


def test_listed_particles_keep_their_species():
    """Hot species that leave the window between sorts are listed and pushed
    with their own charge-to-mass ratio."""
    out = []
    for deposit in ("global", "tiled"):
        print("listed", deposit, flush=True)
        with qa.Region(34, 20, 18, DX, DX, DX, 0.5 * DX, precision="fp64", deposit=deposit, sort_every=0,
                       sort_fallback=0.0, ion_cmr=(0.5, 0.25)) as r:
            rec = _species((34, 20, 18), (2, 2, 2, 2), 5)
            rec[:, 3:6] *= 20
            rec[:, 7] = np.where(rec[:, 7] == 1 / 1836, 0.5, np.where(rec[:, 7] == 1 / 3672, 0.25, rec[:, 7]))
            r.add_records(rec)
            r.init_boundaries()
            d = r.step(8, diag=True)
            if deposit == "tiled":
                assert r.fallback_fraction() > 0.01
            out.append((r.get_fields(), d))
    for a, b in zip(out[1][0], out[0][0]):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
    for a, b in zip(out[1][1], out[0][1]):
        for k in ("energy_e", "energy_p", "energy_ion"):
            assert abs(a[k] - b[k]) <= 1e-11 * abs(b[k])
