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


def _vacuum(capacity):
    """400 electrons at rest, and a pair from vacuum in each of 1728 cells
    (rate x volume x dt = 4e7 at E = E_s)."""
    n, ne = 16, 400
    r = qa.Region(n, n, n, DX, DX, DX, 0.25 * DX, solver="five_point", pusher="vay", precision="fp64", qed=True,
                  e_s=2000.0, q_vac=1e-9, seed=5, capacity=capacity)
    E = np.zeros((n, n, n, 3))
    E[..., 0] = 2000.0
    r.set_fields(E, np.zeros_like(E))
    pos = np.random.default_rng(6).uniform(5, 9, (3, ne))
    r.add_particles(qa.ELECTRON, *pos, *np.zeros((3, ne)), np.full(ne, -1e-9))
    r.init_boundaries()
    return r


def test_step_without_room_moves_nothing():
    """The slots hold the photons of the electrons that were there (400), not
    those of the pairs born as well (3856 leptons)."""
    print("step failure, born pairs", flush=True)
    with _vacuum(3000) as r:
        before, fields = r.particles(qa.ELECTRON)[0], r.get_fields()
        with pytest.raises(qa.QuillError, match="capacity"):
            r.step(1)
        assert (r.particles(qa.ELECTRON)[0][:len(before)] == before).all()
        assert r.count(qa.PHOTON) == 0
        for a, b in zip(r.get_fields(), fields):
            assert (a == b).all()


# slots for every photon before the pairs are counted (8000), and only after
@pytest.mark.parametrize("capacity", [8000, 0])
def test_every_lepton_is_pushed_once(capacity):
    print(f"born pairs {capacity}", flush=True)
    with _vacuum(capacity) as r:
        d = r.step(1, diag=True)[0]
        ue, up = (r.particles(s)[0][:, 3:6] for s in (qa.ELECTRON, qa.POSITRON))
    assert d["n_e"] == len(ue) == 2128 and d["n_p"] == len(up) == 1728
    dt = 0.25 * DX
    # from rest, or born with half a step of the opposite sign; those that
    # emitted a photon recoiled
    recoiled = 0
    for u, want in ((ue[:400], -1.0), (ue[400:], -0.5), (up, 0.5)):
        recoiled += (~np.isclose(u[:, 0], want * 2000.0 * dt, rtol=1e-9, atol=0)).sum()
        assert np.abs(u[:, 1:]).max() == 0
    assert recoiled == d["n_ph"] < 2128
