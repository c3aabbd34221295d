"""Path walks on both sides of the number of live paths below which a step takes the paths to their
ends: one call and many small ones give the same light paths bit for bit."""
import numpy as np
import pytest

from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 65536, 65537, 131101])
@pytest.mark.parametrize("depth", [0, 7])
def test_light_path_batches(ctx, n, depth):
    objs, _ = S.random_field(n_objects=30, seed=4)
    sc = W.Scene(ctx, objs)
    maxv = depth + 3
    whole, counts = sc.light_paths(depth, 5, 2, 100, n, maxv)
    step = 9001
    for p in list(range(0, n, step))[-4:] + [0]:
        m = min(step, n - p)
        part, c = sc.light_paths(depth, 5, 2, 100 + p, m, maxv)
        assert np.array_equal(c, counts[p:p + m])
        keep = np.arange(maxv)[None, :] < c[:, None]
        assert np.array_equal(part[keep].tobytes(), whole[p:p + m][keep].tobytes())
