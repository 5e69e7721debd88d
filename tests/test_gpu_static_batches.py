"""xt_render_static over one and several batches: even shares of the samples, the
last one smaller, and of the pixels."""
import numpy as np
import pytest
import torch

from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


# one batch; shares of the samples; of the pixels
@pytest.mark.parametrize("w,h,spp", [(201, 199, 11), (1501, 997, 7), (2311, 2111, 1)])
@pytest.mark.parametrize("make", [scenes.cornell, lambda w, h: scenes.heightfield(48, w, h)])
def test_static_batches_equal_rounds(make, w, h, spp):
    print(f"[gpu] static batches {w}x{h}x{spp}", flush=True)
    sc = api.Scene(api.Device(0), make(w, h))
    kw = dict(seed=3, max_depth=4, spp_offset=5)
    out = torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    sc.render_static(out.data_ptr(), w, h, spp, **kw)
    sc.set_counting(True)
    assert np.array_equal(out.cpu().numpy(), sc.render(w, h, spp, **kw))
