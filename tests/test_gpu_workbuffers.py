"""Work buffers that a context keeps between calls: calls of changing kinds and sizes, two contexts and
two threads give the films of fresh contexts, and small and large films read back alike."""
import threading

import numpy as np
import pytest

from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


def _ppm(ctx, sc, cam, seed):
    film = W.Film(ctx, cam["width"], cam["height"])
    W.render_ppm(sc, cam, film, 3, 4, seed, 0.05)
    return film.read()["sum"]


def test_changing_calls(ctx):
    want = {}
    sizes = [(9, 7), (40, 30), (24, 24), (41, 30), (9, 7)]
    for w, h in sizes:
        c = W.Context(0)
        objs, cam = S.cornell(k=2, width=w, height=h)
        want[w, h] = _ppm(c, W.Scene(c, objs), cam, 7)
    for k, (w, h) in enumerate(sizes):  # the same in one context, other calls between
        objs, cam = S.cornell(k=2, width=w, height=h)
        sc = W.Scene(ctx, objs)
        assert np.array_equal(_ppm(ctx, sc, cam, 7), want[w, h]), (w, h)
        film = W.Film(ctx, w, h)
        (W.render_bdpt if k % 2 else lambda *a: W.render_vcm(*a, 0.03))(sc, cam, film, 2, 3, 1)
        assert np.isfinite(film.read()["sum"]).all()


def test_two_threads():
    """Two threads, a context each, calls in parallel: no buffer is shared."""
    objs, cam = S.cornell(k=2, width=33, height=21)
    c = W.Context(0)
    want = [_ppm(c, W.Scene(c, objs), cam, s) for s in range(2)]
    got, err = [[], []], []

    def work(t):
        try:
            mine = W.Context(0)
            sc = W.Scene(mine, objs)
            for _ in range(6):
                got[t].append(_ppm(mine, sc, cam, t))
        except Exception as e:  # reported below: an assertion in a thread is lost
            err.append(e)

    ts = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not err
    assert all(np.array_equal(f, want[t]) for t in range(2) for f in got[t])


@pytest.mark.parametrize("width,height", [(1, 1), (295, 296), (296, 296)])  # the last is past the pinned buffer
def test_film_read(ctx, width, height):
    rng = np.random.default_rng(width)
    state = {k: rng.normal(size=3 * width * height).astype(np.float32) for k in ("sum", "comp", "sumsq")}
    film = W.Film(ctx, width, height)
    assert not film.read()["mean"].any()
    film.write(dict(state, passes=3))
    got = film.read()
    for k in state:
        assert np.array_equal(got[k], state[k])
    assert np.array_equal(got["mean"], state["sum"] * (np.float32(1) / np.float32(3)))
    mean = np.zeros(3 * width * height, np.float32)
    W._check(W.lib().wr_film_read(film.h, W._p(mean), None, None, None, None), ctx.h)
    assert np.array_equal(mean, got["mean"])
    film.clear()
    assert film.read()["passes"] == 0 and not film.read()["sumsq"].any()


def test_grid_outlives_context():
    c = W.Context(0)
    g = W.HashGrid.from_points(c, np.random.default_rng(1).random((500, 3)), 0.1, 64)
    c.close()
    g.close()
