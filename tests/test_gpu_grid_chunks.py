"""Hash-grid queries that a workgroup answers chunk by chunk: ranges around the deferral limit and the
chunk size, chunks that are out of reach, partly in reach, coincident, or cut by the cell's ends, and
points at the rim of the radius.  Counts and lists equal the oracle's, order included."""
import numpy as np
import pytest

from oracle import oracle as O
from walkray_amd import _lib as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_cells", [(2048, 1), (2049, 1), (2303, 1), (2305, 1), (9001, 1), (9001, 3)])
def test_crowded_buckets(ctx, n, n_cells):
    rng = np.random.default_rng(n + n_cells)
    pos = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    pos[: n // 3] = 0.25                                        # a coincident heap
    pos[n // 3: n // 2] = np.sort(pos[n // 3: n // 2], axis=0)  # chunks far apart from each other
    r = np.float32(0.125)
    pos[n // 2: n // 2 + 200, :] = 0.5
    pos[n // 2: n // 2 + 200, 0] += r * np.nextafter(np.float32(1), rng.choice([-9, 9], 200).astype(np.float32))
    q = np.concatenate([rng.uniform(0, 1, (150, 3)), np.full((3, 3), 0.25), np.full((3, 3), 0.5), pos[-60:],
                        rng.uniform(-1, 2, (20, 3))]).astype(np.float32)
    g, o = W.HashGrid.from_points(ctx, pos, float(r), n_cells), O.HashGrid(pos, float(r), n_cells)
    cap = 8 * n if n_cells > 1 else 700
    counts, idx = g.query(q, cap)
    want, oidx = o.query(q, cap)
    assert np.array_equal(counts, want)
    for k in range(len(q)):
        m = min(int(want[k]), cap)
        assert np.array_equal(idx[k, :m], oidx[k, :m]), k
