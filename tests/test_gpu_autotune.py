"""xt_scene_autotune on renders whose paths are followed in one launch, which
have no launch shape to tune, and on renders of bounce rounds."""
import numpy as np
import pytest

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


def test_walked_size_keeps_the_shapes():
    dev = api.Device(0)
    for make in (scenes.cornell, scenes.material_zoo):
        sc = api.Scene(dev, make(128, 128))
        kw = dict(seed=3, max_depth=8)
        first = sc.autotune(128, 128, 2, **kw)   # the shapes of a new scene
        for w, h, spp in [(128, 128, 8), (256, 256, 4), (1, 1, 1), (64, 64, 64)]:   # 262,144 paths are the most walked
            print(f"[gpu] autotune, walked {w}x{h}x{spp}", flush=True)
            for rep in range(4):
                assert sc.autotune(w, h, spp, **kw) == first
        tuned = sc.autotune(513, 512, 1, **kw)   # above it: rounds
        print(f"[gpu] autotune, queued: {tuned}", flush=True)
        assert tuned[0] in (2, 4, 5, 6, 7, 8) and tuned[1] in (2, 4, 8)
        assert all(sc.autotune(256, 256, 4, **kw) == tuned for rep in range(4))
        film = sc.render(513, 512, 1, **kw)
        sc.set_counting(True)
        assert np.array_equal(film, sc.render(513, 512, 1, **kw))


def test_guided_size_is_tuned():
    """Guided renders go in rounds at every size."""
    print("[gpu] autotune, guided", flush=True)
    sc = api.Scene(api.Device(0), scenes.cornell(64, 64))
    sc.guide_init(seed=3)
    kw = dict(seed=3, max_depth=4, flags=api.XT_FLAG_GUIDE)
    ref = sc.render(64, 64, 2, **kw)
    tb, sb = sc.autotune(64, 64, 2, **kw)
    assert tb in (2, 4, 5, 6, 7, 8) and sb in (2, 4, 8)
    assert np.array_equal(ref, sc.render(64, 64, 2, **kw))
