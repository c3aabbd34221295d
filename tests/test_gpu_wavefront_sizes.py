"""Wavefront films at the numbers of live paths where its trace stage changes the paths per wave
(a unit of 1, 2, 4, ... 64 paths), starts to draw units from its counters, and where an iteration
takes its paths to their ends: bit-identical to the megakernel's films."""
import numpy as np
import pytest

from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp,slots", [
    (1, 1, 1, 0), (96, 64, 1, 0), (5, 1229, 1, 0), (193, 97, 1, 0), (384, 256, 1, 0), (391, 503, 1, 0),
    (512, 256, 1, 0), (43691, 3, 1, 0),  # the most paths taken to their ends at once, and one more
    (391, 503, 2, 0),        # 393,346 paths: more full units than the resident waves
    (701, 467, 4, 0),        # 1.3M paths: units from the counters, two at a time
    (200, 150, 3, 20000),    # a pool smaller than a pass
])
@pytest.mark.parametrize("nee", [False, True])
def test_paths_per_wave(ctx, width, height, spp, slots, nee):
    objs, cam = S.random_field(n_objects=40, seed=5, width=width, height=height)
    sc = W.Scene(ctx, objs)
    films = []
    for mode in (W.WR_MEGAKERNEL, W.WR_WAVEFRONT):
        film = W.Film(ctx, width, height)
        for k in range(2):  # two calls: the counters are left ready for the next
            W.render(sc, cam, film, spp, 6, 99, mode, wave_slots=slots if mode == W.WR_WAVEFRONT else 0, nee=nee)
        films.append(film.read())
    for k in ("sum", "comp", "sumsq"):
        assert np.array_equal(films[0][k].view(np.uint32), films[1][k].view(np.uint32)), k


@pytest.mark.parametrize("nee", [False, True])
def test_small_pool_is_refilled(ctx, nee):
    """A pool much smaller than a pass takes new paths as others end; only the last are taken to their ends
    in one iteration.  (An iteration that ended every path of a full pool would make one turn per pool of
    paths and wait for the longest path each time; a path of the Cornell box has three segments or more.)"""
    objs, cam = S.cornell(k=2, width=400, height=300)
    slots = 16384
    st = W.render(W.Scene(ctx, objs), cam, W.Film(ctx, 400, 300), 2, 8, 5, W.WR_WAVEFRONT, wave_slots=slots, nee=nee)
    turns = -(-st["paths"] // slots)
    assert st["iterations"] > 1.5 * turns, (st["iterations"], turns)
