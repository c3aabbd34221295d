"""The reference box test where its proof on the exit face is not conclusive or has no face to stand
on: rays to the corners and edges of the meshes (and of their boxes), along the axes, with zero and
tiny direction components, long directions, and from origins in the planes of the boxes."""
import numpy as np
import pytest

from oracle import oracle as O
from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu


def _edge_rays(objs, seed):
    rng = np.random.default_rng(seed)
    v = np.concatenate([np.asarray(ob["verts"], np.float32).reshape(-1, 3) for ob in objs])
    lo, hi = v.min(0), v.max(0)
    a, b = v[rng.integers(len(v), size=(2, 6000))]
    target = np.concatenate([a, (a + b) * np.float32(0.5)])       # corners, and points of edges and faces
    o = (lo + (hi - lo) * rng.random((len(target), 3)) * 1.5).astype(np.float32)
    d = target - o
    for axis in range(3):                                         # in the plane of a box face, and along it
        sel = rng.random(len(o)) < 0.15
        o[sel, axis] = target[sel, axis]
        d[sel, axis] = rng.choice(np.array([0, -0.0, 1e-31, -1e-31, 1e-30, 1e-20], np.float32), sel.sum())
    keep = np.abs(d).max(1) > 1e-6
    o, d = o[keep], d[keep]
    n = np.linalg.norm(d, axis=1, keepdims=True)
    scale = rng.choice([1.0, 1.0, 1e-3, 37.0], size=(len(d), 1))  # directions need not be unit vectors
    return np.concatenate([o, (d / n * scale).astype(np.float32)], axis=1).astype(np.float32)


@pytest.mark.parametrize("name", ["cornell", "field", "heightfield"])
def test_rays_at_box_edges(ctx, name):
    objs = {"cornell": lambda: S.cornell(k=2, width=8, height=8)[0],
            "field": lambda: S.random_field(n_objects=20, seed=3)[0],
            "heightfield": lambda: [S.heightfield(65, seed=4)]}[name]()
    rays = _edge_rays(objs, 11)
    hits, ref = W.Scene(ctx, objs).closest_hit(rays), O.Scene(objs).intersect(rays)
    assert np.array_equal(hits["prim"], ref["prim"])
    assert np.array_equal(hits["t"].view(np.uint32), ref["t"].view(np.uint32))
    assert 0.1 < (ref["prim"] != O.NONE).mean()
