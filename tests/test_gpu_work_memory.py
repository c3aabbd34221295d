"""The work buffers that a context keeps, at the end of device memory (wr_ctx_limit_work_memory): every
allocation of the context gets the unused ones' memory before it fails."""
import numpy as np
import pytest

from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


def _fill(ctx, sc, cam):
    """Leaves the buffers of a BidirectionalPathTracer call unused."""
    film = W.Film(ctx, cam["width"], cam["height"])
    W.render_bdpt(sc, cam, film, 2, 4, 1)


def _wavefront(sc, cam, film, spp):
    W.render(sc, cam, film, spp, 4, 1, W.WR_WAVEFRONT, wave_slots=65536)


# What is prepared before the device is full, and the call whose first allocation finds it full.
def _render(ctx, sc, cam):
    film = W.Film(ctx, cam["width"], cam["height"])
    return lambda: _wavefront(sc, cam, film, 3)  # the path pool


def _window(ctx, sc, cam):
    film = W.Film(ctx, cam["width"], cam["height"])
    _wavefront(sc, cam, film, 1)
    return lambda: _wavefront(sc, cam, film, 8)  # a larger sample window in the same pool


def _moving(ctx, sc, cam):
    objs, _, motions = S.cornell_moving(k=2, width=cam["width"], height=cam["height"])
    m = W.Scene(ctx, objs, build=False)
    for obj, (t0, t1, a, b) in motions.items():
        m.set_motion(obj, t0, t1, a, b)
    m.build()
    film = W.Film(ctx, cam["width"], cam["height"])
    return lambda: _wavefront(m, cam, film, 2)  # the pass's scene


def _autotune(ctx, sc, cam):
    rays = ctx.to_device(np.ones((999, 6), np.float32))
    return lambda: sc.autotune_closest_hit(rays, 999)


CALLS = {
    "render": _render,
    "window": _window,
    "moving": _moving,
    "autotune": _autotune,
    "scene": lambda ctx, sc, cam: lambda: W.Scene(ctx, S.cornell(k=1)[0]),
    "server": lambda ctx, sc, cam: lambda: W.Server(ctx, path_slots=65536),
    "alloc": lambda ctx, sc, cam: lambda: ctx.alloc(1 << 20),
}


@pytest.mark.parametrize("call", sorted(CALLS))
def test_unused_buffers_are_given_back(call):
    ctx = W.Context(0)
    objs, cam = S.cornell(k=2, width=96, height=80)
    sc = W.Scene(ctx, objs)
    run = CALLS[call](ctx, sc, cam)
    _fill(ctx, sc, cam)
    held = sum(ctx.work_memory())
    unused = ctx.work_memory()[1]
    assert unused > 32 << 20
    ctx.limit_work_memory(held)  # the device has no more than the context holds
    try:
        kept = run()  # noqa: F841
        assert ctx.work_memory()[1] < unused
    finally:
        ctx.limit_work_memory(0)


def test_limit_is_reported():
    """Past the limit a call fails with an error, and the next one within it succeeds."""
    ctx = W.Context(0)
    objs, cam = S.cornell(k=2, width=96, height=80)
    sc = W.Scene(ctx, objs)
    film = W.Film(ctx, 96, 80)
    ctx.limit_work_memory(1 << 20)
    with pytest.raises(Exception, match="memory"):
        W.render_bdpt(sc, cam, film, 2, 4, 1)
    with pytest.raises(Exception, match="memory"):
        W.Film(ctx, 1000, 1000)
    ctx.limit_work_memory(0)
    W.render_bdpt(sc, cam, film, 2, 4, 1)
    assert film.read()["sum"].any()


def test_jobs_and_films_hold_their_size():
    """A served job holds what its budget counts and a film its three arrays, also where larger unused
    buffers would fit them."""
    ctx = W.Context(0)
    objs, cam = S.cornell(k=2, width=96, height=80)
    sc = W.Scene(ctx, objs)
    server = W.Server(ctx, path_slots=1 << 16)
    sid = server.add_scene(sc)
    cam2 = dict(cam, width=64, height=64)
    sizes = []
    for _ in range(2):  # the second job takes the first one's buffers
        bufs = [W.Film(ctx, 80 + 10 * k, 80) for k in range(12)]  # a ladder of unused sizes
        del bufs
        _fill(ctx, sc, cam)
        jid = server.submit(sid, cam2, 200, 4, 1)
        server.step()
        used = ctx.work_memory()[0]
        while server.step():
            pass
        assert abs(used - server.status(jid)["device_bytes"]) <= 2 * 256
        sizes.append(sum(ctx.work_memory()))
        server.release(jid)
    assert sizes[0] == sizes[1]
    assert ctx.work_memory()[0] == 0
    film = W.Film(ctx, 70, 64)
    assert 0 <= ctx.work_memory()[0] - 3 * 12 * 70 * 64 <= 256
    film.close()


@pytest.mark.parametrize("kind", ["bdpt", "vcm"])
@pytest.mark.parametrize("depth", [1, 5, 32])
def test_prefixes_without_room(kind, depth):
    """The prefixes of the sub-path records are 56 B beside a record's 72: an image whose records fit renders
    without room for them all.  Sums of up to 4,096 nonnegative terms in any order agree to 4096 * 2^-24."""
    objs, cam = S.cornell(k=2, width=96, height=80)
    table = 56 * 2 * (depth + 3) * 96 * 80 * 2
    args, films, held = () if kind == "bdpt" else (0.03,), [], 0
    for room in (None, 0.6, 0.05):  # of the table
        ctx = W.Context(0)
        sc, film = W.Scene(ctx, objs), W.Film(ctx, 96, 80)
        if room is not None:
            ctx.limit_work_memory(int(held - (1 - room) * table))
        getattr(W, f"render_{kind}")(sc, cam, film, 2, depth, 5, *args)
        if room is None:
            held = sum(ctx.work_memory())
        else:
            assert sum(ctx.work_memory()) <= held - (1 - room) * table
        films.append(film.read()["sum"])
    assert films[0].any()
    for f in films[1:]:
        assert np.allclose(f, films[0], rtol=2.5e-4, atol=1e-30)
