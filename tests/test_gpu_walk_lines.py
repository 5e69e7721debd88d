"""Which renders are followed in one launch (one extend launch, counted) and
which go in rounds: by paths, depth cap, normal maps and whether the scene is
open -- under a sky, with less surface than its bounds' own.  Either way the
film is that of the rounds."""
import numpy as np
import pytest

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


def _sky(d):
    d.env = scenes.Env(True, (1.0, 1.0, 1.0))
    return d


def _nmap(d):
    d.materials = [scenes.microfacet_nmap(m) if m.type == scenes.MAT_DIFFUSE else m for m in d.materials]
    return d


def _field(w, h):
    return scenes.heightfield(48, w, h)


def _canyon(w, h):
    return scenes.heightfield(48, w, h, amplitude=1.0)


def _no_sky(w, h):
    d = _field(w, h)
    d.env = scenes.Env()
    return d


def _plane(w, h):
    return scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32))


K = 1 << 16
# scene, depth cap, most paths walked
CASES = {
    "room": (lambda w, h: scenes.occluded_room(w, h, n_tris=2000), 4, 4 * K),
    "room_under_sky": (lambda w, h: _sky(scenes.occluded_room(w, h, n_tris=2000)), 4, 4 * K),
    "cornell_under_sky": (lambda w, h: _sky(scenes.cornell(w, h)), 4, 4 * K),
    "canyon": (_canyon, 4, 4 * K),
    "field": (_field, 4, 10 * K),
    "field_no_sky": (_no_sky, 4, 4 * K),
    "plane": (_plane, 4, 8 * K),
    "cornell_uncapped": (scenes.cornell, 0, 10 * K),
    "cornell_nmap_uncapped": (lambda w, h: _nmap(scenes.cornell(w, h)), 0, 5 * K),
    "empty_sky": (lambda w, h: scenes.SceneDesc(objects=[], materials=[scenes.diffuse(0.5)], env=scenes.Env(True, (1.0, 1.0, 1.0)),
                                                camera=scenes.cornell(w, h).camera), 4, 4 * K),
}


@pytest.mark.parametrize("kind", list(CASES))
def test_line(kind):
    make, depth, most = CASES[kind]
    sc = api.Scene(api.Device(0), make(512, 512))
    kw = dict(seed=2, max_depth=depth)
    for w, h, walked in ((512, most // 512, True), (most // 512 + 1, 512, False)):
        print(f"[gpu] walk lines: {kind} {w}x{h}", flush=True)
        film = sc.render(w, h, 1, **kw)
        assert (sc.stats()["extend_launches"] == 1) == walked or kind == "empty_sky"
        sc.set_counting(True)
        assert np.array_equal(film, sc.render(w, h, 1, **kw))
        sc.set_counting(False)
