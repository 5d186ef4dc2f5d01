"""Second pieces of crossing paths kept by their lane in the tiled push: FP32
against the oracle where few and where most particles cross a face per step,
some two or three, in one round per workgroup and in many, tiles in halves (180
tiles); and tiles at the box's corners, where the staged nodes are clamped."""
import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


@pytest.mark.parametrize("shape,ppc,sigma", [((8, 8, 8), 1, 0.02), ((9, 16, 17), 3, 0.5), ((24, 17, 16), 40, 0.02),
                                             ((24, 17, 16), 40, 3.0), ((41, 48, 40), 3, 0.3)])
def test_crossings_match_oracle(shape, ppc, sigma):
    rec, ids = oracle.synth_plasma(*shape, ppc, 0.02, sigma, 7)
    rec = rec.astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(3)
    E, B = (rng.uniform(-0.05, 0.05, shape + (3,)).astype(np.float32).astype(np.float64) for _ in range(2))
    o = oracle.Oracle(*shape, DX, DX, DX, 0.5 * DX, solver=oracle.FDTD, pusher=oracle.BORIS)
    o.field(oracle.E)[:] = E
    o.field(oracle.B)[:] = B
    o.add_particles(rec, ids)
    o.init_boundaries()
    o.step(1)
    print(f"crossings {shape} {ppc} {sigma}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision="fp32", deposit="tiled") as r:
        r.set_fields(E, B)
        r.add_records(rec)
        r.init_boundaries()
        r.step(1)
        J = r.get_fields()[2]
    # one step: each node sums at most some thousands of FP32 terms of relative
    # error 2^-22 (weights) whose magnitudes are bounded by the largest |J|
    ref = o.field(oracle.J)
    assert np.linalg.norm(J - ref) <= 2e-5 * np.linalg.norm(ref)
    assert np.abs(J - ref).max() <= 2e-4 * np.abs(ref).max()
