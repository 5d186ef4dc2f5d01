"""Rows by id: ids that two live particles share are refused, whether in one
block of rows or in two."""
import numpy as np
import pytest

import quill_amd as qa

pytestmark = pytest.mark.gpu

DX = 0.05 * 2 * np.pi


# 64 MiB hold 1118481 rows and their marks
@pytest.mark.parametrize("n,first,second", [(2, 0, 1), (300, 3, 299), (1118482, 0, 1118481), (1118482, 1118480, 1118479)])
def test_shared_ids_are_refused(n, first, second):
    print(f"shared ids {n} {first} {second}", flush=True)
    pos = 1 + 13 * np.random.default_rng(2).random((3, n))
    with qa.Region(17, 17, 17, DX, DX, DX, 0.5 * DX, track_ids=True) as r:
        ids = np.arange(n, dtype=np.int32)
        ids[second] = ids[first]
        r.add_particles(qa.ELECTRON, *pos, *np.zeros((3, n)), np.full(n, -1e-6), ids=ids)
        with pytest.raises(qa.QuillError, match="share"):
            r.rows_by_id(qa.ELECTRON, n)
        # no ids given: all are 0
        r.add_particles(qa.POSITRON, *pos[:, :2], *np.zeros((3, 2)), np.full(2, 1e-6))
        with pytest.raises(qa.QuillError, match="share"):
            r.rows_by_id(qa.POSITRON, 2)
