"""Paths that do not end.  Without a depth cap a render whose paths go on past
some 64 Ki vertices fails, whether they are queued or followed in one launch,
and leaves the film as it was.  Two parallel mirrors hold the paths; a
roulette that starts near the limit and lets none through ends every path soon
after it in any case."""
import numpy as np
import pytest

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

LAST = 65534   # the last vertex a path may go on from the one before


def _mirrors(width, height, fov):
    s = scenes.SceneDesc(name="mirrors")
    m = s.add_material(scenes.Material(scenes.MAT_SPEC_REFL))
    for z in (-1.0, 1.0):
        v, i = scenes.quad((-100, -100, z), (100, -100, z), (100, 100, z), (-100, 100, z))
        s.objects.append(scenes.ObjectDesc(v, i, material=m))
    s.env = scenes.Env(has_sky=True, sky=(0.5, 0.75, 1.0))
    s.camera = scenes.Camera(scenes.translate(30.0, -20.0, 0.0)[0], fov, height / width)   # looks along +z
    return api.Scene(api.Device(0), s)


def _kw(rr_start, max_depth=0):
    return dict(seed=2, max_depth=max_depth, rr_start=rr_start, rr_prob=1e-30)


def _render(sc, w, h, film, kw, counting=False):
    """The error's text, or None."""
    sc.set_counting(counting)
    try:
        sc.render(w, h, 1, film=film, **kw)
        return None
    except api.XtError as e:
        return str(e)
    finally:
        sc.set_counting(False)


@pytest.mark.parametrize("counting", [False, True])   # followed in one launch, queued
def test_limit_is_the_same_walked_and_queued(counting):
    w, h = 8, 4
    sc = _mirrors(w, h, 2e-6)
    for rr_start in (LAST, LAST + 1):
        print(f"[gpu] path limit: {rr_start} vertices counting={counting}", flush=True)
        film = np.full((h, w, 3), 3.0, np.float32)
        err = _render(sc, w, h, film, _kw(rr_start), counting)
        assert np.all(film == 3.0)   # nothing reaches the sky
        if rr_start == LAST:
            assert err is None and sc.stats()["extension_rays"] == w * h * LAST
        else:
            assert err is not None and "did not drain" in err


def test_render_after_a_failed_one():
    w, h = 8, 4
    sc = _mirrors(w, h, 2e-6)
    print("[gpu] path limit: a render after a failed one", flush=True)
    assert _render(sc, w, h, np.zeros((h, w, 3), np.float32), _kw(LAST + 1)) is not None
    kw = dict(seed=2, max_depth=5, camera=_mirrors(w, h, 3.0).desc.camera)   # steep rays reach the sky
    film = sc.render(w, h, 4, **kw)
    sc.set_counting(True)
    assert film.max() > 0.0 and np.array_equal(film, sc.render(w, h, 4, **kw))


def test_limit_in_the_walked_tail():
    """Most paths leave in the first hundreds of rounds; the others are followed from the queue."""
    w, h = 1024, 768
    sc = _mirrors(w, h, 0.2)
    for rr_start in (2000, LAST + 1):
        print(f"[gpu] path limit: tail, {rr_start} vertices", flush=True)
        film = np.full((h, w, 3), 3.0, np.float32)
        err = _render(sc, w, h, film, _kw(rr_start))
        if rr_start == 2000:
            assert err is None and film.max() > 3.0
        else:
            assert err is not None and "did not drain" in err and np.all(film == 3.0)


def test_depth_cap_above_the_limit():
    w, h = 8, 4
    print("[gpu] path limit: a depth cap above it", flush=True)
    sc = _mirrors(w, h, 2e-6)
    film = np.full((h, w, 3), 3.0, np.float32)
    assert _render(sc, w, h, film, _kw(LAST + 100, max_depth=70000)) is None
    assert sc.stats()["extension_rays"] == w * h * (LAST + 100) and np.all(film == 3.0)


def test_ray_counts_after_a_failed_render():
    """The rays of the failed render are not counted again by the next one."""
    w, h = 8, 4
    sc = _mirrors(w, h, 2e-6)
    print("[gpu] path limit: ray counts after a failed render", flush=True)
    assert _render(sc, w, h, np.zeros((h, w, 3), np.float32), _kw(LAST + 1)) is not None
    sc.render(w, h, 1, **_kw(100))
    assert sc.stats()["extension_rays"] == w * h * 100
