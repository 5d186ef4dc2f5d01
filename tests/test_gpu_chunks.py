"""The tiled push with tiles cut into parts (grids of few tiles): FP64 against
the global deposit on the same inputs, at one tile, at the most tiles that
are cut and one layer more, from less than one part per tile to many."""
import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


@pytest.mark.parametrize("shape,ppc", [((8, 8, 8), 1), ((8, 8, 8), 300), ((17, 9, 10), 40), ((64, 32, 32), 1),
                                       ((64, 32, 32), 9), ((66, 32, 31), 9)])
def test_parts_match_global_deposit(shape, ppc):
    rec, ids = oracle.synth_plasma(*shape, ppc, 0.02, 0.3, 11)
    rng = np.random.default_rng(2)
    E, B = rng.uniform(-0.1, 0.1, shape + (3,)), rng.uniform(-0.1, 0.1, shape + (3,))
    out = []
    for deposit in ("global", "tiled"):
        print(f"chunks {shape} {ppc} {deposit}", flush=True)
        with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision="fp64", deposit=deposit, sort_every=2) as r:
            r.set_fields(E, B)
            r.add_records(rec)
            r.init_boundaries()
            d = r.step(5, diag=True)
            out.append((r.get_fields(), d[-1]["n_e"], d[-1]["energy_e"]))
    for a, b in zip(out[1][0], out[0][0]):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    assert out[1][1] == out[0][1]
    assert abs(out[1][2] - out[0][2]) <= 1e-12 * abs(out[0][2])


@pytest.mark.parametrize("shape,ppc", [((72, 48, 40), 6), ((72, 48, 40), 3), ((64, 64, 64), 6), ((65, 64, 64), 6)])
def test_halves_match_global_deposit(shape, ppc):
    """Tiles in halves (270 and 512 tiles, with and without enough particles)
    and one layer more than are cut."""
    test_parts_match_global_deposit(shape, ppc)
