"""Be interpolated from B on its own (init_boundaries), at random fields: both
forms of the kernel (FP64 above 2^20 cells stages B in LDS) against plain
sums, at edges of the blocks and on planes dealt to the XCDs in bands."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


def expected(B):
    n = B.shape[:3]
    planes = sum(np.isin(np.arange(m), (0, m - 1)).astype(int).reshape([-1 if x == a else 1 for x in range(3)])
                 for a, m in enumerate(n))
    out = np.zeros_like(B)
    for c in range(3):
        F, cnt = B[..., c], np.ones(n)
        for a in range(3):
            s = 1 if a == c else -1
            F2, c2 = np.zeros(n), np.zeros(n)
            to = [slice(None)] * 3
            of = [slice(None)] * 3
            to[a], of[a] = (slice(None, -1), slice(1, None)) if s == 1 else (slice(1, None), slice(None, -1))
            F2[tuple(to)], c2[tuple(to)] = F[tuple(of)], cnt[tuple(of)]
            F, cnt = F + F2, cnt + c2
        out[..., c] = np.where(planes < 2, F * np.where(cnt == 8, 0.125, 0.25), 0.0)
    return out


@pytest.mark.parametrize("precision,shape", [("fp32", (5, 5, 5)), ("fp32", (7, 129, 128)), ("fp32", (9, 13, 67)),
                                             ("fp64", (6, 5, 63)), ("fp64", (64, 128, 128)), ("fp64", (65, 128, 128)),
                                             ("fp64", (120, 93, 97))])
def test_be_matches_plain_sums(precision, shape):
    rng = np.random.default_rng(sum(shape))
    print(f"Be {shape} {precision}", flush=True)
    with qa.Region(*shape, DX, DX, DX, 0.5 * DX, precision=precision) as r:
        r.set_fields(rng.normal(size=shape + (3,)), rng.normal(size=shape + (3,)))
        r.init_boundaries()
        _, B, _, Be = r.get_fields()
    want = expected(B)
    # sums of eight numbers and one multiplication by a power of two
    tol = 8 * (2.0 ** -24 if precision == "fp32" else 2.0 ** -53) * np.abs(B).max()
    assert np.abs(Be - want).max() <= tol
