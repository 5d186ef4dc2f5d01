"""A step that finds no room for its particles: the call fails and leaves the
state of the last finished step, wherever in the call that step was."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi
DTF = {"fdtd": 0.5, "ndfx": 0.5, "five_point": 0.25}


def _radiating(solver, precision, source):
    """Photon slots for exactly one step of 300 leptons that all may emit."""
    n, ne, nph = 12, 300, 700
    rng = np.random.default_rng(11)
    r = qa.Region(n, n, n, DX, DX, DX, DTF[solver] * DX, solver=solver, pusher="vay", precision=precision, qed=True,
                  e_s=4e5, seed=3, capacity=ne + nph)
    E, B = rng.uniform(-20, 20, (2, n, n, n, 3))
    B[..., 2] += 1000.0
    r.set_fields(E, B)
    for s, m, q in ((qa.ELECTRON, ne, -1e-9), (qa.PHOTON, nph, 1e-9)):
        r.add_particles(s, *rng.uniform(5, 7, (3, m)), np.full(m, 5000.0), np.zeros(m), np.zeros(m), np.full(m, q))
    if source:
        w = 0.2 * 2 * np.pi
        r.add_laser_source(0, 3, 5.0, 2.0, w, w, w, 3 * DX, x1=-1.0)
    r.init_boundaries()
    return r


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("solver,source", [("fdtd", False), ("ndfx", True), ("five_point", False)])
def test_fields_after_a_failed_call(solver, source, precision):
    got = []
    for calls in ((4,), (1, 1)):   # the second step fails
        print(f"step failure {solver} {precision} {calls}", flush=True)
        with _radiating(solver, precision, source) as r:
            for n in calls[:-1]:
                r.step(n)
            with pytest.raises(qa.QuillError, match="capacity"):
                r.step(calls[-1])
            got.append(r.get_fields())
    # the same operations in the same order, but for the order of the current's
    # terms: 300 leptons of 1e-9 against fields of 1e3, so a last bit may tip
    tol = 4 * np.finfo(np.float32 if precision == "fp32" else np.float64).eps
    for k in (0, 1, 3):
        assert np.abs(got[0][k] - got[1][k]).max() <= tol * np.abs(got[1][k]).max()
