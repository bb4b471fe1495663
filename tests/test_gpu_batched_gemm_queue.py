"""The batched GEMM's work queues: every tile is done once whether a segment has
fewer items than workgroups, more, or nearly all there are, also when the call
is replayed.  Integer data, so the products are exact."""
import numpy as np
import pytest

from test_gpu_batched_gemm import _run

pytestmark = pytest.mark.gpu

BATCHES = {
    "fewer_than_workgroups": [(20 + 3 * i, 70 - i, 5) for i in range(13)],
    "one_segment_has_most": [(2000, 1500, 9)] + [(10 + i, 12, 6) for i in range(30)],
    "two_rounds": [(33 + i % 3, 40, 5) for i in range(900)],
    "many_rounds": [(64 - i % 40, 65 + i % 30, 4) for i in range(2500)],
    "single": [(1, 1, 1)],
}


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("name", BATCHES)
def test_every_tile_once(oba, dt, name):
    rng = np.random.default_rng(1)
    draw = lambda r, c: np.asfortranarray(rng.integers(-3, 4, (r, c)).astype(dt))
    probs = [{"m": m, "n": n, "k": k, "a": draw(m, k), "b": draw(k, n), "c": draw(m, n)} for m, n, k in BATCHES[name]]
    want = [p["c"].copy(order="F") for p in probs]
    for _ in range(3):   # C accumulates, so a tile done twice shows
        _run(oba, dt, 0, 0, probs, 1.0, 1.0)
        for p, w in zip(probs, want):
            w += p["a"] @ p["b"]
            assert np.array_equal(p["c"], w), (p["m"], p["n"], p["k"])
