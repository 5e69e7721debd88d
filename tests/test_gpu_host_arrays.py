"""Calls on host arrays give what the same calls on device arrays give, on both
sides of the size from which rays are copied to the device, and with the kept
copies taken by films of other sizes in between."""
import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-1.2, 1.2, (n, 3))
    rays[:, 3] = np.where(rng.random(n) < 0.5, np.inf, rng.uniform(0.1, 3.0, n))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    return rays


def test_host_queries_equal_device_queries():
    sc = api.Scene(api.Device(0), scenes.material_zoo(64, 64))
    for n in (1, 63, 1001, 32768, 32769, 5, 40000):
        print(f"[gpu] host query of {n} rays", flush=True)
        rays = _rays(n, n)
        dev = torch.from_numpy(rays).to("cuda:0")
        hits = torch.zeros((n, 4), dtype=torch.float32, device="cuda:0")
        occ = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
        torch.cuda.synchronize()
        sc.trace_closest_dev(dev.data_ptr(), n, hits.data_ptr())
        sc.trace_any_dev(dev.data_ptr(), n, occ.data_ptr())
        host = np.ascontiguousarray(sc.trace_closest(rays))
        assert host.tobytes() == hits.cpu().numpy().tobytes()
        assert np.array_equal(np.asarray(sc.trace_any(rays)).astype(np.uint8), occ.cpu().numpy())


@pytest.mark.parametrize("f64", [False, True])
def test_host_films_equal_device_films(f64):
    dev = api.Device(0)
    sc = api.Scene(dev, scenes.cornell(64, 64))
    for w, h, spp in [(64, 40, 1), (900, 700, 1), (1, 1, 1), (300, 200, 2)]:
        print(f"[gpu] host film {w}x{h}x{spp} f64={f64}", flush=True)
        start = np.random.default_rng(w).random((h, w, 3))
        film = start.astype(np.float64 if f64 else np.float32)
        ref = torch.from_numpy(film.copy()).to("cuda:0")
        torch.cuda.synchronize()
        kw = dict(seed=2, max_depth=4)
        sc.render(w, h, spp, film=film, f64=f64, **kw)
        sc.render_device(ref.data_ptr(), w, h, spp, f64=f64, **kw)
        assert np.array_equal(film, ref.cpu().numpy())


def test_host_queries_of_several_threads():
    """Each thread its own scene: one query at a time has the mapped buffer, the others copy."""
    import threading
    dev, n = api.Device(0), 3000
    jobs = []
    for k in range(4):
        sc, rays = api.Scene(dev, scenes.material_zoo(64, 64)), _rays(n, k)
        jobs.append((sc, rays, sc.trace_closest(rays).tobytes(), sc.trace_any(rays).tobytes()))
    print("[gpu] host queries of four threads", flush=True)
    wrong = []

    def work(sc, rays, hits, occ):
        for _ in range(20):
            if sc.trace_closest(rays).tobytes() != hits or sc.trace_any(rays).tobytes() != occ:
                wrong.append(sc)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
