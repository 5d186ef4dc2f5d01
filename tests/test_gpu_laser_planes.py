"""Laser-source corrections at the edges of their kernel's tiles: the source
planes at the ends of their ranges and next to each other, transverse sizes
around the 64 x 4 columns of a workgroup, two tilted pulses on one side;
vacuum, FP64, against the oracle's source (1e-10)."""
import math

import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

TWO_PI = 2 * math.pi
DX = 0.05 * TWO_PI
SOLVERS = {"fdtd": (oracle.FDTD, 0.5), "ndfx": (oracle.NDFX, 0.5), "five_point": (oracle.FIVE_POINT, 0.35)}


def pulse(x0, x1, tilt, phi):
    w = 0.35 * TWO_PI
    return np.array([1.0, 0.4, w, w, 0.9 * w, x0, 1, x1, 0.3, tilt, -tilt, 1, phi, 0.0, 0.0, 0.0])


@pytest.mark.parametrize("shape,planes", [((20, 9, 65), (2, 18)), ((24, 5, 64), (18, 6)), ((22, 13, 67), (10, 11)),
                                          ((22, 8, 130), (9, 13)), ((16, 17, 20), (2, None)), ((16, 12, 63), (None, 14))])
@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_source_planes_match_oracle(solver, shape, planes):
    code, dtf = SOLVERS[solver]
    nx = shape[0]
    o = oracle.Oracle(*shape, DX, DX, DX, dtf * DX, solver=code, pusher=oracle.VAY)
    print(f"source planes {solver} {shape} {planes}", flush=True)
    with qa.Region(*shape, DX, DX, DX, dtf * DX, solver=solver, pusher="vay", precision="fp64") as r:
        for side, plane in enumerate(planes):
            if plane is None:
                continue
            mid = plane * DX
            for L in (pulse(mid - 0.5 if side == 0 else mid + 0.5, -1.0 if side == 0 else 1.0, 0.0, 0.0),
                      pulse(mid, -1.0 if side == 0 else 1.0, 0.15, 0.4)):
                o.laser_source(L, side, plane)
                r.add_laser_source(side, plane, *L[:11], phi=L[12])
        o.init_boundaries()
        r.init_boundaries()
        o.step(12)
        r.step(12)
        E, B, _, _ = r.get_fields()
    for name, a, b in zip("EB", (E, B), (o.field(oracle.E), o.field(oracle.B))):
        assert np.abs(b).max() > 0.05
        err = np.abs(a - b).max() / np.abs(b).max()
        print(f"{name}: {err:.2e}", flush=True)
        assert err < 1e-10, name


@pytest.mark.parametrize("plasma", [False, True])
@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_one_call_equals_single_steps(solver, plasma):
    """Half steps of B taken in pairs inside a call, with the sources' corrections
    and the field energy in between, against calls of one step: FP64, sums of
    the same terms in another order."""
    shape = (24, 11, 66)
    dtf = SOLVERS[solver][1]
    rec, ids = oracle.synth_plasma(*shape, 1, 0.02, 0.1, 17)
    out = []
    for calls in ((1,) * 14, (14,), (3, 11)):
        print(f"calls {solver} plasma {plasma} {calls}", flush=True)
        with qa.Region(*shape, DX, DX, DX, dtf * DX, solver=solver, pusher="vay", precision="fp64", sort_every=4) as r:
            if plasma:
                r.add_records(rec)
            for side, plane in ((0, 3), (1, 19)):
                L = pulse(plane * DX, -1.0 if side == 0 else 1.0, 0.15, 0.4)
                r.add_laser_source(side, plane, *L[:11], phi=L[12])
            r.init_boundaries()
            en = [d["energy_f"] for n in calls for d in r.step(n, diag=True)]
            out.append((r.get_fields(), en))
    assert out[0][1][-1] > 10 * out[0][1][1] > 0
    for f, en in out[1:]:
        np.testing.assert_allclose(en, out[0][1], rtol=1e-12)
        for a, b in zip(f, out[0][0]):
            assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
