"""Window kernel from lengths with keys out of order: windows whose bags lie in one run of the lengths, in two (staged by
one wave, both fronts in one sum) and in more, on both sides of the 256 bags that one wave stages, and calls in which a
wave takes several rounds; against the CPU oracle, bit for bit."""
import numpy as np
import pytest

import oracle as O
from helpers import bits_equal
from test_tbe_gpu import _from_lengths, build

pytestmark = pytest.mark.gpu

ORDERS = {"reversed": [5, 4, 3, 2, 1, 0], "pairs": [4, 5, 0, 1, 7, 8], "gap": [0, 1, 2, 4, 5, 6], "last first": [8, 0, 1, 2, 3, 4]}


@pytest.mark.parametrize("order", list(ORDERS))
@pytest.mark.parametrize("B", [1, 7, 60, 129, 300])
@pytest.mark.parametrize("window", [64, 150, 256, 257])
@pytest.mark.parametrize("idt", [np.int32, np.int64])
def test_runs(tuning, order, B, window, idt):
    tuning(balanced=1, window=window, fused_scan=1)
    rng = np.random.default_rng(B + window)
    order = ORDERS[order]
    T, K = len(order), max(order) + 1
    specs = [((O.INT4 if idt == np.int32 else O.INT8), 90 + t, 64) for t in range(T)]
    tbe, store = build(rng, specs, list(range(T)), O.SUM, O.FP16, 16)
    lengths = rng.choice([0, 1, 2, 5, 30], K * B).astype(idt)
    starts = np.concatenate([[0], np.cumsum(lengths)])
    ids = rng.integers(0, 90, int(starts[-1])).astype(idt)
    # the oracle takes the features' bags in feature order
    picks = np.concatenate([np.arange(p * B, (p + 1) * B) for p in order])
    seg = np.concatenate([np.arange(starts[q], starts[q + 1]) for q in picks])
    offsets = np.zeros(T * B + 1, dtype=idt)
    offsets[1:] = np.cumsum(lengths[picks])
    want = O.tbe_forward(store, list(range(T)), B, ids[seg], offsets, None, O.SUM, O.FP16)
    assert bits_equal(_from_lengths(tbe, ids, lengths, None, B, feature_positions=order), want) == 0
