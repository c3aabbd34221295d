"""Ray batches around the sizes where wr_closest_hit and wr_closest_hit_noself change their launch:
one lane per ray over few or many waves, and the persistent kernel with its counters.  Every ray of a
batch is compared with the oracle bit for bit (the batch repeats a base set of rays)."""
import numpy as np
import pytest

from oracle import oracle as O
from walkray_amd import _lib as W
from walkray_amd import scenes as S

pytestmark = pytest.mark.gpu

BASE = 20011  # not a multiple of 64, so that a repeated ray meets other lanes and units
SMALL_MAX = {False: 1 << 19, True: 1 << 21}  # the largest one-launch batch, without and with NoSelf


@pytest.fixture(scope="module")
def field(ctx):
    objs, cam = S.random_field(n_objects=24, seed=8, width=120, height=90)
    sc, osc = W.Scene(ctx, objs), O.Scene(objs)
    lo, hi = S.scene_bounds(objs)
    rays = np.concatenate([S.pinhole_rays(cam), S.incoherent_rays(BASE - 120 * 90, lo, hi, seed=6)])
    first = osc.intersect(rays)
    ok = first["prim"] != O.NONE
    path = rays.copy()
    path[ok, :3] += rays[ok, 3:] * first["t"][ok, None]
    path[:, 3:] = S.incoherent_rays(BASE, lo, hi, seed=7)[:, 3:]
    contact = np.where(ok, first["obj"], O.NONE).astype(np.uint32)
    inside = np.where(np.arange(BASE) % 3 == 0, contact, O.NONE).astype(np.uint32)
    return sc, rays, first, path, inside, contact, osc.intersect(path, inside, contact, noself=True)


def _check(hits, ref, idx, label):
    assert np.array_equal(hits["prim"], ref["prim"][idx]), label
    hit = hits["prim"] != O.NONE
    for k in ("t", "b1", "b2"):
        got, want = hits[k].view(np.uint32), ref[k][idx].view(np.uint32)
        sel = slice(None) if k == "t" else hit
        assert np.array_equal(got[sel], want[sel]), f"{label}: {k}"


@pytest.mark.parametrize("n", [1, 65, 6144, 6145, 98305, 393217, SMALL_MAX[False], SMALL_MAX[False] + 1, 1100003])
def test_closest_hit_sizes(field, n):
    sc, rays, ref = field[:3]
    idx = np.arange(n) % BASE
    _check(sc.closest_hit(rays[idx]), ref, idx, f"{n} rays")


@pytest.mark.parametrize("n", [1, 6145, 196609, SMALL_MAX[True], SMALL_MAX[True] + 77])
def test_noself_sizes(field, n):
    sc, path, inside, contact, ref = (field[k] for k in (0, 3, 4, 5, 6))
    idx = np.arange(n) % BASE
    _check(sc.closest_hit_noself(path[idx], inside[idx], contact[idx]), ref, idx, f"{n} NoSelf rays")


@pytest.mark.parametrize("tuning", [(1, 1, 1, 4, 64), (64, 65, 0, 16, 4096), (16, 32, 3, 8, 128)])
def test_persistent_launch_choices(field, tuning):
    """Every launch configuration of the persistent kernel gives the same hits (few and many units
    per workgroup, every unit through the counter, stripes cut by the end of the batch)."""
    sc, rays, ref = field[:3]
    idx = np.arange(700001) % BASE
    sc.set_closest_hit_tuning(*tuning)
    try:
        for _ in range(2):  # the counters are left zeroed for the next call
            _check(sc.closest_hit(rays[idx]), ref, idx, str(tuning))
        _check(sc.closest_hit(rays[:333], counters=True)[0], ref, idx[:333], f"{tuning} counted")
    finally:
        sc.set_closest_hit_tuning(16, 32)


@pytest.mark.parametrize("n_objects", [24, 100])  # on both sides of the tree size where NoSelf batches change their order
@pytest.mark.parametrize("n", [49152, 49153, 65537, 98305, 196608, 196609])
def test_noself_orders(ctx, field, n_objects, n):
    """The one-launch NoSelf batch at the sizes where its lanes per wave and the order of its rays change.
    The larger scene's rays are compared with the same rays in small batches."""
    idx = np.arange(n) % BASE
    if n_objects == 24:
        sc, path, inside, contact, ref = (field[k] for k in (0, 3, 4, 5, 6))
        _check(sc.closest_hit_noself(path[idx], inside[idx], contact[idx]), ref, idx, f"{n} NoSelf rays")
        return
    objs, _ = S.random_field(n_objects=n_objects, seed=8)
    assert sum(len(o["tris"]) for o in objs) > 81920
    sc, path, contact = W.Scene(ctx, objs), field[3], np.full(BASE, O.NONE, np.uint32)
    base = sc.closest_hit_noself(path, contact, contact)
    _check(sc.closest_hit_noself(path[idx], contact[idx], contact[idx]), base, idx, f"{n} NoSelf rays")
