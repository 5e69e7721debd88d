"""Count-driven batches against the same renders in rounds with fetches counted:
per-item graphs too large to be walked, and walked windows of several scenes
whose waves start full, so that a wave's last paths move to its first lanes
with the scenes they belong to."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu

ENV = api.XT_FLAG_ENV_NEE
SCENES = {
    "cornell": (scenes.cornell, {}),
    "zoo": (scenes.material_zoo, {}),
    "field": (lambda w, h: scenes.heightfield(48, w, h), {"flags": ENV}),
    "zoo_sorted": (scenes.material_zoo, {"flags": api.XT_FLAG_SORT_MATERIALS}),
}
PLANE = (lambda w, h: scenes.displaced_plane(grid=48, width=w, height=h, normal_map_size=64, sky_size=(64, 32)), {"flags": ENV})


def _counted(sc, w, h, spp, kw):
    sc.set_counting(True)
    film = sc.render(w, h, spp, **kw)
    sc.set_counting(False)
    return film


@pytest.mark.parametrize("w,h,spp", [(513, 512, 1), (823, 797, 1), (641, 383, 5)])   # just above what is walked, closed and open, and more
@pytest.mark.parametrize("kind", [*SCENES, "plane"])
def test_item_graphs_equal_rounds(monkeypatch, kind, w, h, spp):
    monkeypatch.setenv("XITILS_AMD_BATCH", "items")
    print(f"[gpu] cursor rounds: {kind} {w}x{h}x{spp}", flush=True)
    make, kw = PLANE if kind == "plane" else SCENES[kind]
    sc, kw = api.Scene(api.Device(0), make(w, h)), {"seed": 4, "max_depth": 5, "spp_offset": 2, **kw}
    ref = torch.from_numpy(_counted(sc, w, h, spp, kw))
    film = torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0")   # one film: one graph, replayed
    for rep in range(3):
        film.zero_()
        torch.cuda.synchronize()
        api.render_batch([(sc, w, h, spp, (film.data_ptr(), False), kw)])
        assert torch.equal(film.cpu(), ref)


def _windows(plane):
    """Scenes of odd sizes, 200 k to 250 k paths in all."""
    dev, jobs, ref = api.Device(0), [], []
    makes = [*SCENES.values(), PLANE] if plane else list(SCENES.values())
    for k, (make, kw) in enumerate(makes * 2):
        w, h, spp = 75 + 8 * k, 117 - 8 * k, 3
        sc, kw = api.Scene(dev, make(w, h)), {"seed": 5 + k, "max_depth": 7, **kw}
        jobs.append((sc, w, h, spp, None, kw))
        ref.append(_counted(sc, w, h, spp, kw))
    paths = sum(j[1] * j[2] * j[3] for j in jobs)
    assert (1 << 17) < paths <= 1 << 18
    for rep in range(2):
        films, _ = api.render_batch(jobs)
        for a, b in zip(films, ref):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("plane", [False, True])
def test_full_waves_of_several_scenes(plane):
    print(f"[gpu] cursor rounds: walked window of several scenes, normal maps={plane}", flush=True)
    _windows(plane)


def test_several_walked_windows():
    """The same batch in windows of 200,000 paths (read once per process)."""
    print("[gpu] cursor rounds: several walked windows", flush=True)
    here = os.path.dirname(os.path.abspath(__file__))
    code = f"import sys; sys.path[:0] = [{os.path.dirname(here)!r}, {here!r}]; import test_gpu_cursor_rounds as t; t._windows(False); t._windows(True)"
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, XITILS_AMD_PATHS="200000"), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
