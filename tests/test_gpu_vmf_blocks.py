"""The EM fit's two forms (a wave per sample set, a block per set) give the
same bits: the same sets are fitted by few (blocks) and among many others
(more sets than the block form takes)."""
import numpy as np
import pytest

from xitils_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lobes", [1, 2, 6, 7, 12, 16])
def test_block_and_wave_fits_are_the_same_bits(lobes):
    print(f"[gpu] vmf fit: {lobes} lobes", flush=True)
    rng = np.random.default_rng(lobes)
    sizes = [2, 63, 64, 65, 0, 1, 1023, 1024, 1025, 3001]   # rounds of 64 around the block's waves and batches
    mean = rng.normal(size=(len(sizes), 3))
    x = [m + 0.6 * rng.normal(size=(n, 3)) for m, n in zip(mean, sizes)]
    x = np.concatenate([v / np.linalg.norm(v, axis=1, keepdims=True) for v in x]).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    iu = rng.random((len(sizes), 2 * lobes)).astype(np.float32)
    dev = api.Device(0)
    enc, steps = api.vmf_fit(dev, lobes, x, off, iu)
    many = 1025 - len(sizes)   # one set more than the block form takes; the others are empty
    off2 = np.concatenate([off, np.full(many, off[-1], np.uint32)])
    enc2, steps2 = api.vmf_fit(dev, lobes, x, off2, np.concatenate([iu, np.zeros((many, 2 * lobes), np.float32)]))
    assert np.array_equal(steps, steps2[:len(sizes)])
    assert np.array_equal(enc.view(np.uint32), enc2[:len(sizes)].view(np.uint32))
