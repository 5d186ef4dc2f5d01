"""QED steps whose reserved capacity holds the worst case only after the pairs
born from vacuum are counted, against steps that have room for all at once;
and pairs born from vacuum in every step, pushed in the step of their birth."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("capacity", [0, 1000])
def test_charge_is_conserved_at_tight_capacity(capacity, precision):
    n, ne, nph = 12, 200, 300   # 512 cells may bear a pair: 200 + 512 + 300 > 1000
    rng = np.random.default_rng(4)
    print(f"qed capacity {capacity} {precision}", flush=True)
    with qa.Region(n, n, n, DX, DX, DX, 0.25 * DX, solver="five_point", pusher="vay", precision=precision, qed=True,
                   e_s=4e5, seed=3, capacity=capacity) as r:
        B = np.zeros((n, n, n, 3))
        B[..., 2] = 1000.0
        r.set_fields(np.zeros_like(B), B)
        for s, m, q in ((qa.ELECTRON, ne, -1e-6), (qa.PHOTON, nph, 1e-6)):
            pos = rng.uniform(5, 7, (3, m))
            r.add_particles(s, *pos, np.full(m, 5000.0), np.zeros(m), np.zeros(m), np.full(m, q))
        r.init_boundaries()
        d = r.step(4, diag=True)
    for x in d:
        assert x["n_e"] - x["n_p"] == ne          # pairs come in pairs, and none has left yet
        assert x["n_ph"] > 0 and x["n_nonfinite"] == 0
    assert d[-1]["n_ph"] + d[-1]["n_p"] > nph     # photons were emitted


def test_pairs_from_vacuum_are_pushed_at_once():
    """In a uniform E along x every pair gains u = +- E dt (less the half step
    it is born with) in the step it is born in; those that emit a photon in
    the same push recoil, one lepton per photon."""
    n = 16
    E = np.zeros((n, n, n, 3))
    E[..., 0] = 2000.0
    with qa.Region(n, n, n, DX, DX, DX, 0.25 * DX, solver="five_point", pusher="vay", precision="fp64", qed=True,
                   e_s=2000.0, q_vac=1e-9, seed=5) as r:
        r.set_fields(E, np.zeros_like(E))
        print("vacuum pairs", flush=True)
        d = r.step(1, diag=True)[0]
        ue, up = (r.particles(s)[0][:, 3:6] for s in (qa.ELECTRON, qa.POSITRON))
    assert d["n_e"] == d["n_p"] == len(ue) == len(up) > 100
    dt = 0.25 * DX
    # born with +E dt / 2, pushed by -E dt (electrons); positrons the other way round
    recoiled = 0
    for u, sign in ((ue, -1), (up, 1)):
        ok = np.isclose(u[:, 0], sign * 0.5 * 2000.0 * dt, rtol=1e-9, atol=0)
        recoiled += (~ok).sum()
        assert np.abs(u[:, 1:]).max() == 0
    assert recoiled == d["n_ph"] < len(ue)
