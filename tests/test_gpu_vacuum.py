"""Steps without charged particles: Be interpolated once per call, the half
steps of B run in pairs, the zero current skipped.  One call of many steps,
many calls of one step and the oracle give the same fields and energies, on
planes below and above the size where sweeps are dealt to the XCDs in bands;
and a plasma that leaves the box is followed by the same steps."""
import math

import numpy as np
import pytest

import oracle
import quill_amd as qa

pytestmark = pytest.mark.gpu

TWO_PI = 2 * math.pi
DX = 0.05 * TWO_PI
SOLVERS = {"fdtd": (oracle.FDTD, 0.5), "ndfx": (oracle.NDFX, 0.5), "five_point": (oracle.FIVE_POINT, 0.35)}


def pulse(shape):
    w = 0.2 * TWO_PI
    return dict(a0y=1.0, a0z=0.5, xsigma=w, ysigma=w, zsigma=w, x0=0.5 * shape[0] * DX, x1=-1.0, phase=0.3, phi=0.4)


# 65 blocks of 256 cells per plane, 63 of them, one partly filled
@pytest.mark.parametrize("shape", [(12, 130, 127), (12, 127, 126), (21, 9, 13)])
@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_paired_half_steps(solver, shape):
    code, dtf = SOLVERS[solver]
    o = oracle.Oracle(*shape, DX, DX, DX, dtf * DX, solver=code, pusher=oracle.BORIS)
    o.laser_cos(**pulse(shape))
    o.init_boundaries()
    o.step(7)
    for precision, tight, bar in (("fp64", 1e-14, 1e-10), ("fp32", 2e-6, 1e-4)):
        got = []
        for calls in ((7,), (1,) * 7, (2, 5)):
            print(f"vacuum {solver} {shape} {precision} {calls}", flush=True)
            with qa.Region(*shape, DX, DX, DX, dtf * DX, solver=solver, pusher="boris", precision=precision) as r:
                r.init_laser_cos(**pulse(shape))
                r.init_boundaries()
                en = [d["energy_f"] for n in calls for d in r.step(n, diag=True)]
                got.append((r.get_fields(), en))
        for f, en in got[1:]:
            for a, b in zip(f, got[0][0]):
                assert np.abs(a - b).max() <= tight * np.abs(b).max()
            np.testing.assert_allclose(en, got[0][1], rtol=1e-12 if precision == "fp64" else 1e-6)
        for a, b in zip(got[0][0], (o.field(oracle.E), o.field(oracle.B), o.field(oracle.J), o.field(oracle.BE))):
            assert np.abs(a - b).max() <= bar * max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_plasma_that_leaves(solver):
    shape = (20, 14, 17)
    code, dtf = SOLVERS[solver]
    n = 40
    rng = np.random.default_rng(4)
    rec = np.zeros((n, 8))
    rec[:, 0] = shape[0] - 3 + rng.random(n)
    rec[:, 1:3] = 4 + 6 * rng.random((n, 2))
    rec[:, 3] = 50.0
    rec[:, 6], rec[:, 7] = -0.01, -1
    o = oracle.Oracle(*shape, DX, DX, DX, dtf * DX, solver=code, pusher=oracle.BORIS)
    o.add_particles(rec, np.arange(n, dtype=np.int32))
    o.init_boundaries()
    with qa.Region(*shape, DX, DX, DX, dtf * DX, solver=solver, pusher="boris", precision="fp64", sort_every=2) as r:
        r.add_records(rec)
        r.init_boundaries()
        for steps in (3, 3, 1, 4):
            print(f"leaving {solver} {steps}", flush=True)
            o.step(steps)
            r.step(steps)
            E, B, J, Be = r.get_fields()
            for name, a, b in (("E", E, oracle.E), ("B", B, oracle.B), ("Be", Be, oracle.BE)):
                b = o.field(b)
                assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max(), name
        assert r.count(qa.ELECTRON) == 0 and not J.any()
