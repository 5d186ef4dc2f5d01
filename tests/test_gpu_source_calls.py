"""Laser sources in one call of many steps and in many calls of one step: the
same operations in the same order, so the same bits of every field, on both
sides of the box and with planes that lie next to each other."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi
DTF = {"fdtd": 0.5, "ndfx": 0.5, "five_point": 0.25}


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("solver", sorted(DTF))
@pytest.mark.parametrize("shape,planes", [((21, 9, 13), (3,)), ((24, 70, 66), (4, 20)), ((16, 8, 130), (7, 8))])
def test_calls_do_not_change_the_fields(shape, planes, solver, precision):
    w = 0.4 * 2 * np.pi
    got = []
    for calls in ((8,), (1,) * 8, (3, 5)):
        print(f"source calls {shape} {solver} {precision} {calls}", flush=True)
        with qa.Region(*shape, DX, DX, DX, DTF[solver] * DX, solver=solver, precision=precision) as r:
            for side, plane in enumerate(planes):
                r.add_laser_source(side, plane, 1.5, 0.7, w, w, w, (plane - 1 + 2 * side) * DX,
                                   x1=-1.0 if side == 0 else 1.0, phase=0.4 + side, phi=0.3)
            r.init_boundaries()
            en = [d["energy_f"] for n in calls for d in r.step(n, diag=True)]
            got.append((r.get_fields(), en))
    assert np.abs(got[0][0][0]).max() > 0.1
    for fields, en in got[1:]:
        for a, b in zip(fields, got[0][0]):
            assert (a == b).all()
        np.testing.assert_allclose(en, got[0][1], rtol=1e-6 if precision == "fp32" else 1e-12, atol=1e-9 * max(en))
