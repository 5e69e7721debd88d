"""Renders whose paths are followed to their ends in one launch (small batches
and windows, the last rounds of large ones) give the bits and the ray totals of
the queued kernels, which a scene renders with while it counts fetches."""
import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

KINDS = {
    "cornell": (lambda w, h: scenes.cornell(w, h), {}),
    "zoo_roulette_only": (lambda w, h: scenes.material_zoo(w, h), {"max_depth": 0}),
    "zoo_naive": (lambda w, h: scenes.material_zoo(w, h), {"integrator": 1}),
    "field": (lambda w, h: scenes.heightfield(48, w, h), {"flags": api.XT_FLAG_ENV_NEE}),
    "plane": (lambda w, h: scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32)),
              {"flags": api.XT_FLAG_ENV_NEE}),
}


def _scene(kind, w, h):
    make, kw = KINDS[kind]
    kw = {"seed": 3, "max_depth": 6, **kw}
    return api.Scene(api.Device(0), make(w, h)), kw


# one path, a ragged wave, more than one path a wave, more than a chunk, full waves
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (13, 5, 1), (67, 45, 1), (131, 97, 3), (257, 193, 5)])
@pytest.mark.parametrize("kind", list(KINDS))
def test_walked_equals_queued(kind, w, h, spp):
    print(f"[gpu] walk: {kind} {w}x{h}x{spp}", flush=True)
    sc, kw = _scene(kind, w, h)
    film = sc.render(w, h, spp, **kw)
    st = sc.stats()
    sc.set_counting(True)
    ref = sc.render(w, h, spp, **kw)
    sr = sc.stats()
    assert np.array_equal(film, ref)
    for key in ("camera_rays", "extension_rays", "shadow_rays"):
        assert st[key] == sr[key], key
    sc.set_counting(False)
    if kw["max_depth"] > 0:
        out = torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        sc.render_static(out.data_ptr(), w, h, spp, **kw)
        assert np.array_equal(out.cpu().numpy(), ref)


# more paths than are walked from the camera: the first rounds are queued, the rest walked
@pytest.mark.parametrize("kind", ["cornell", "zoo_roulette_only", "plane"])
def test_queued_rounds_then_walked(kind):
    w, h, spp = 641, 383, 3
    print(f"[gpu] walk after queued rounds: {kind}", flush=True)
    sc, kw = _scene(kind, w, h)
    film = sc.render(w, h, spp, f64=True, **kw)
    st = sc.stats()
    sc.set_counting(True)
    assert np.array_equal(film, sc.render(w, h, spp, f64=True, **kw))
    sr = sc.stats()
    for key in ("camera_rays", "extension_rays", "shadow_rays"):
        assert st[key] == sr[key], key


def test_walked_batch_equals_single_renders():
    print("[gpu] walk: batch window over five scenes", flush=True)
    dev, jobs, ref = api.Device(0), [], []
    for k, (make, kw) in enumerate(KINDS.values()):
        w, h, spp = 17 + 30 * k, 31 + 7 * k, 1 + k
        sc = api.Scene(dev, make(w, h))
        kw = {"seed": 5 + k, "max_depth": 7, **kw}
        kw["max_depth"] = kw["max_depth"] or 9
        jobs.append((sc, w, h, spp, None, kw))
        sc.set_counting(True)
        ref.append(sc.render(w, h, spp, **kw))
        sc.set_counting(False)
    for rep in range(3):   # replays and fresh captures
        films, _ = api.render_batch(jobs)
        for a, b in zip(films, ref):
            assert np.array_equal(a, b)
