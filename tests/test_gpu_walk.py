"""Path walks on both sides of the number of live paths below which a step takes the paths to their
ends: one call and many small ones give the same light paths bit for bit."""
import time

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


def _bright_box():
    """A closed box of albedo 0.99 with a small light under its ceiling: paths of hundreds of scatters."""
    return [S.box((0, 0, 0), (1, 1, 1), S.DIFFUSE, (0.99, 0.99, 0.99), inward=True),
            S.quad((0.5, 0.999, 0.5), (0.1, 0, 0), (0, 0, 0.1), (0, -1, 0), S.EMISSIVE, (5.0, 5.0, 5.0))]


def test_long_walks(ctx):
    """More than 65,536 paths alive after the last list step: the same light paths as in batches of few,
    which are taken to their ends from the start."""
    sc, n, depth, maxv = W.Scene(ctx, _bright_box()), 131101, 60, 63
    whole, counts = sc.light_paths(depth, 5, 2, 100, n, maxv)
    assert (counts > 33 + 2).sum() > 65536
    for p in (0, 60000, n - 9001):
        part, c = sc.light_paths(depth, 5, 2, 100 + p, 9001, maxv)
        assert np.array_equal(c, counts[p:p + 9001])
        keep = np.arange(maxv)[None, :] < c[:, None]
        assert np.array_equal(part[keep].tobytes(), whole[p:p + 9001][keep].tobytes())


@pytest.mark.parametrize("n", [1000, 70000])
def test_path_limit_costs_no_launches(ctx, n):
    """The time of a call follows its paths, not the limit on their length: light paths in the open field,
    where none has 40 scatters, with limits of 40 and 1,000 (two launches a step made that 5 ms of 0.3)."""
    sc = W.Scene(ctx, S.random_field(n_objects=30, seed=4)[0])

    def best(depth):
        buf = ctx.alloc(64 * n * (depth + 3)), ctx.alloc(4 * n)
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            W._check(W.lib().wr_light_paths(ctx.h, sc.h, depth, 5, 2, 100, n, depth + 3, buf[0].ptr, buf[1].ptr), ctx.h)
            t.append(time.perf_counter() - t0)
        return min(t), buf[1].download(np.uint32, n)

    (short, c0), (long, c1) = best(40), best(1000)
    assert np.array_equal(c0, c1) and c0.max() < 42
    assert long < 2.5 * short + 2e-4, (short, long)
