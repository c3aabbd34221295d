"""Connections at the image sizes where the lanes per wave change, with queues that hold them all, few
of them (a reservation then ends past the queue) or one.  All contributions are nonnegative, so sums of
up to 4,096 of them in any order agree to 4096 * 2^-24 relative."""
import numpy as np
import pytest

from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bdpt", "vcm"])
@pytest.mark.parametrize("width,height,spp", [(1, 1, 1), (63, 65, 1), (128, 64, 1), (91, 181, 1), (256, 256, 1),
                                              (256, 257, 2)])
def test_queue_sizes(ctx, kind, width, height, spp):
    objs, cam = S.cornell(k=2, width=width, height=height)
    sc, args = W.Scene(ctx, objs), () if kind == "bdpt" else (0.03,)
    sums = []
    for queue in (0, 1000, 1):
        film = W.Film(ctx, width, height)
        getattr(W, f"render_{kind}")(sc, cam, film, spp, 6, 17, *args, queue=queue)
        sums.append(film.read()["sum"])
    assert sums[0].any() or width == 1
    for s in sums[1:]:
        assert np.allclose(s, sums[0], rtol=2.5e-4, atol=1e-30)
