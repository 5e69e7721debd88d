"""First rounds that make their camera rays where they are traced and shaded give
the bits of the rounds with a queue of camera rays, which a scene renders with
while it counts fetches."""
import numpy as np
import pytest

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

SORT = api.XT_FLAG_SORT_MATERIALS
KINDS = {
    "zoo_sorted": (lambda w, h: scenes.material_zoo(w, h), {"flags": SORT}),
    "plane_sorted": (lambda w, h: scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32)),
                     {"flags": api.XT_FLAG_ENV_NEE | SORT}),
    "zoo_naive": (lambda w, h: scenes.material_zoo(w, h), {"integrator": 1}),
}


@pytest.mark.parametrize("w,h,spp,first", [(641, 383, 3, 0), (1023, 641, 1, 7)])   # ragged last waves and blocks
@pytest.mark.parametrize("kind", list(KINDS))
def test_made_equals_queued_camera_rays(kind, w, h, spp, first):
    print(f"[gpu] camera round: {kind} {w}x{h}x{spp}", flush=True)
    make, kw = KINDS[kind]
    kw = {"seed": 4, "max_depth": 5, "spp_offset": first, **kw}
    sc = api.Scene(api.Device(0), make(w, h))
    film = sc.render(w, h, spp, **kw)
    sc.set_counting(True)
    assert np.array_equal(film, sc.render(w, h, spp, **kw))
