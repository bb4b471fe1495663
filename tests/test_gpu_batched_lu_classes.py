"""Batched LU where size classes share a launch: a problem has the same factors,
pivots and info, bit for bit, whatever batch it comes in (alone it runs with as
many threads as it has rows), in batches that join two, three and four classes
and in one that joins none."""
import numpy as np
import pytest

from test_gpu_batched_lu import _run

pytestmark = pytest.mark.gpu

BATCHES = {
    "four": [1, 8, 33, 64, 65, 100, 128, 129, 200, 256, 257, 400, 512],
    "top_and_bottom": [300, 5, 17, 64],
    "two_middle": [70, 90, 128, 129, 150],
    "lower_two": [20, 64, 65, 100],
    "none_above_one": [128] + [40] * 3000,
}


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("name", BATCHES)
def test_same_bits_in_any_batch(oba, dt, name):
    rng = np.random.default_rng(2)
    mats = [rng.standard_normal((m, m + (i % 3 - 1) * (m > 2))).astype(dt) for i, m in enumerate(BATCHES[name])]
    mats[len(mats) // 2][:, 0] = 0                      # one of them singular
    lds = [a.shape[0] + i % 2 for i, a in enumerate(mats)]
    bufs, pivs, info = _run(oba, dt, mats, lds)
    assert (info != 0).sum() >= 1
    for i in range(min(len(mats), 20)):
        b, p, f = _run(oba, dt, mats[i:i + 1], lds[i:i + 1])
        assert np.array_equal(bufs[i], b[0]) and np.array_equal(pivs[i], p[0]) and info[i] == f[0], mats[i].shape
