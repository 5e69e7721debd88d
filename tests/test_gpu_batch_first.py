"""A device handle's first batch while the default stream is busy: the batch's
chunk cursors are cleared on its own stream, before its first launch."""
import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


def test_first_batch_beside_a_busy_default_stream():
    w, h, spp = 96, 64, 2
    kw = dict(seed=3, max_depth=6)
    desc = scenes.material_zoo(w, h)
    ref = api.Scene(api.Device(0), desc).render(w, h, spp, **kw)
    a = torch.randn(4096, 4096, device="cuda:0")
    (a @ a).sum().item()
    for rep in range(3):
        print(f"[gpu] first batch, default stream busy, {rep}", flush=True)
        sc = api.Scene(api.Device(0), desc)
        films = [torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0") for _ in range(2)]
        torch.cuda.synchronize()
        for _ in range(40):
            b = a @ a
        api.render_batch([(sc, w, h, spp, (f.data_ptr(), False), kw) for f in films])
        for f in films:
            assert np.array_equal(f.cpu().numpy(), ref)
    del b
