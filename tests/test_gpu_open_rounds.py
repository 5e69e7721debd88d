"""Rounds under a sky, whose misses are shaded as they come and whose hits are
collected for whole blocks, give the bits of the rounds shaded in queue order,
which a scene renders with while it counts fetches."""
import numpy as np
import pytest

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

ENV = api.XT_FLAG_ENV_NEE
KINDS = {
    "field": (lambda w, h: scenes.heightfield(48, w, h), {"flags": ENV}),
    "field_no_env_nee": (lambda w, h: scenes.heightfield(48, w, h), {}),
    "field_naive": (lambda w, h: scenes.heightfield(48, w, h), {"integrator": 1}),
    "plane": (lambda w, h: scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32)),
              {"flags": ENV}),
}
# just above what is walked in one launch (the last block of a queue nearly empty), and many rounds of a block
SIZES = [(1024, 641, 1), (1409, 1091, 2)]


@pytest.mark.parametrize("w,h,spp", SIZES)
@pytest.mark.parametrize("kind", list(KINDS))
def test_open_rounds_equal_queue_order(kind, w, h, spp):
    print(f"[gpu] open rounds: {kind} {w}x{h}x{spp}", flush=True)
    make, kw = KINDS[kind]
    kw = {"seed": 6, "max_depth": 9, **kw}
    sc = api.Scene(api.Device(0), make(w, h))
    film = sc.render(w, h, spp, **kw)
    st = sc.stats()
    sc.set_counting(True)
    assert np.array_equal(film, sc.render(w, h, spp, **kw))
    sr = sc.stats()
    for key in ("camera_rays", "extension_rays", "shadow_rays"):
        assert st[key] == sr[key], key


def test_open_batch_equals_single_renders():
    """A window over scenes with and without a sky."""
    w, h, spp = 641, 383, 2
    print(f"[gpu] open rounds: batch of {w}x{h}x{spp}", flush=True)
    dev, jobs, ref = api.Device(0), [], []
    for k, (make, kw) in enumerate([*KINDS.values(), (scenes.cornell, {})]):
        sc = api.Scene(dev, make(w, h))
        kw = {"seed": 7 + k, "max_depth": 5, **kw}
        jobs.append((sc, w, h, spp, None, kw))
        sc.set_counting(True)
        ref.append(sc.render(w, h, spp, **kw))
        sc.set_counting(False)
    films, _ = api.render_batch(jobs)
    for a, b in zip(films, ref):
        assert np.array_equal(a, b)
