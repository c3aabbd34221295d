"""Connections and merges from per-record prefixes (BidirectionalPathTracer, VCMTracer) and photon
throughputs (PhotonMap) at the path lengths where they start and end: one-record sub-paths, paths that
end at the length limit, the longest ones, glass before a light point, and a scene without emitters.
Against the oracle, which sweeps every joined path: the sub-paths are the same up to libm's last ulp,
which can turn a path, so most pixel sums (a share that every row reaches with a margin) agree to 1e-4,
and none is off by its own size while the whole image is within its standard errors."""
import numpy as np
import pytest

from oracle import oracle as O
from walkray_amd import _lib as W
from walkray_amd import render as R
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bdpt", "vcm", "ppm"])
@pytest.mark.parametrize("depth", [0, 1, 2, 32])
def test_path_lengths(ctx, kind, depth):
    objs, cam = S.cornell(k=2, width=23, height=19)
    sc, osc = W.Scene(ctx, objs), O.Scene(objs)
    film = W.Film(ctx, cam["width"], cam["height"])
    spp, args = 12, () if kind == "bdpt" else (0.04,)
    getattr(W, f"render_{kind}")(sc, cam, film, spp, depth, 31, *args)
    g = film.read()
    s, q = getattr(osc, f"render_{kind}")(cam, spp, depth, 31, *args)
    same = np.isclose(g["sum"], s.astype(np.float32), rtol=1e-4, atol=1e-6).mean()
    assert same > 0.5, f"only {same:.3f} of the pixel sums agree"
    mean, se = R.film_stats(g)
    mo = s / spp
    se = np.sqrt(se ** 2 + np.maximum(q / spp - mo * mo, 0) / spp)
    z = np.abs(mean - mo)[se > 0] / se[se > 0]
    assert np.allclose(mean[se == 0], mo[se == 0], rtol=1e-5, atol=1e-5)
    assert z.size == 0 or ((z > 3).mean() <= 0.01 and z.max() <= 6), (z > 3).mean()


@pytest.mark.parametrize("kind", ["bdpt", "vcm"])
def test_no_emitter(ctx, kind):
    """Empty light samples connect to nothing: a black film."""
    objs, cam = S.cornell(k=1, width=16, height=16)
    objs = [dict(o, mat=S.DIFFUSE, params=(0.5, 0.5, 0.5)) if o["mat"] == S.EMISSIVE else o for o in objs]
    film = W.Film(ctx, 16, 16)
    getattr(W, f"render_{kind}")(W.Scene(ctx, objs), cam, film, 2, 4, 1, *([0.05] if kind == "vcm" else []))
    assert not film.read()["sum"].any()
