"""Renders that trace a round's shadow rays in the launch of the next round's
extension rays give the bits and the ray totals of the separate launches, which
a scene renders with while it counts fetches."""
import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

KINDS = {
    "cornell": (lambda w, h: scenes.cornell(w, h), {}),
    "zoo_roulette_only": (lambda w, h: scenes.material_zoo(w, h), {"max_depth": 0}),
    "cornell_depth_1": (lambda w, h: scenes.cornell(w, h), {"max_depth": 1}),
    "field": (lambda w, h: scenes.heightfield(48, w, h), {"flags": api.XT_FLAG_ENV_NEE}),
    "plane": (lambda w, h: scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32)),
              {"flags": api.XT_FLAG_ENV_NEE}),
}


def _scene(kind, w, h):
    make, kw = KINDS[kind]
    return api.Scene(api.Device(0), make(w, h)), {"seed": 3, "max_depth": 6, **kw}


def _separate(sc, w, h, spp, kw):
    sc.set_counting(True)
    film = sc.render(w, h, spp, **kw)
    st = sc.stats()
    sc.set_counting(False)
    return film, st


def _same_rays(a, b):
    for key in ("camera_rays", "extension_rays", "shadow_rays", "extend_launches"):
        assert a[key] == b[key], key


# guided renders are queued at every size: one path, a ragged wave, some blocks
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (13, 5, 1), (67, 45, 2), (131, 97, 3)])
@pytest.mark.parametrize("kind", ["cornell", "cornell_depth_1", "zoo_roulette_only"])
def test_guided_joint_equals_separate(kind, w, h, spp):
    print(f"[gpu] joint: guided {kind} {w}x{h}x{spp}", flush=True)
    sc, kw = _scene(kind, w, h)
    sc.guide_init(seed=3)
    kw["flags"] = kw.get("flags", 0) | api.XT_FLAG_GUIDE
    ref, sr = _separate(sc, w, h, spp, kw)
    assert np.array_equal(sc.render(w, h, spp, **kw), ref)
    _same_rays(sc.stats(), sr)
    if kw["max_depth"] > 0:
        for rep in range(3):   # a captured loop and its replays
            films, _ = api.render_batch([(sc, w, h, spp, None, kw)])
            assert np.array_equal(films[0], ref)


# queued from the camera: even shares, and (12 M paths) chunks
@pytest.mark.parametrize("w,h,spp", [(641, 383, 3), (1409, 1091, 8)])
@pytest.mark.parametrize("kind", list(KINDS))
def test_queued_joint_equals_separate(kind, w, h, spp):
    print(f"[gpu] joint: {kind} {w}x{h}x{spp}", flush=True)
    sc, kw = _scene(kind, w, h)
    ref, sr = _separate(sc, w, h, spp, kw)
    assert np.array_equal(sc.render(w, h, spp, **kw), ref)
    st = sc.stats()
    for key in ("camera_rays", "extension_rays", "shadow_rays"):
        assert st[key] == sr[key], key
    if kw["max_depth"] > 0:
        out = torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        sc.render_static(out.data_ptr(), w, h, spp, **kw)
        assert np.array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("w,h,spp", [(257, 193, 5), (1025, 577, 4)])   # one window of even shares, of chunks
def test_joint_batch_equals_separate_renders(w, h, spp):
    print(f"[gpu] joint: batch of {w}x{h}x{spp}", flush=True)
    dev, jobs, ref = api.Device(0), [], []
    for k, (make, kw) in enumerate(KINDS.values()):
        sc = api.Scene(dev, make(w, h))
        kw = {"seed": 5 + k, "max_depth": 6, **kw}
        kw["max_depth"] = kw["max_depth"] or 9
        jobs.append((sc, w, h, spp, None, kw))
        ref.append(_separate(sc, w, h, spp, kw)[0])
    for rep in range(3):   # replays and fresh captures
        films, _ = api.render_batch(jobs)
        for a, b in zip(films, ref):
            assert np.array_equal(a, b)
