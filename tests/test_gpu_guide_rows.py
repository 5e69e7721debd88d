"""xt_guide_gradient at the edges of the packing blocks (256 samples), of the
gradient kernel's groups (128 samples, a partial row each) and of the rows'
summation, against the bf16 reference."""
import numpy as np
import pytest

import guide_ref as G
from xitils_amd import api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 127, 128, 129, 256, 257, 32768, 32769])
def test_gradient_at_block_edges(n):
    print(f"[gpu] guide gradient n={n}", flush=True)
    sc = api.Scene(api.Device(0), scenes.cornell(32, 32))
    sc.guide_init(seed=3)
    lo, hi = (b.astype(np.float64) for b in sc.guide_bounds())
    P = G.init_params(16)
    sc.guide_set_params(P)
    q, d = G.random_queries(n, lo, hi, 300 + n), G.random_dirs(n, 400 + n)
    w = np.random.default_rng(n).exponential(1.0, n).astype(np.float32)
    g = sc.guide_gradient(q, d, w, 1.0, 4.0)
    gr = G.backward(P, q, d, w, lo, hi, emulate=True, weight_scale=1.0, weight_clip=4.0)
    rel = np.linalg.norm(g - gr) / np.linalg.norm(gr)
    print(f"[gpu]   rel err vs bf16 reference {rel:.2e}", flush=True)
    assert rel <= 2e-2   # the bf16 activations' rounding, as tests/test_guide.py
