"""Window kernel of several launch classes in one launch: every body it holds, and the widths at which its lane groups
change, against the CPU oracle, bit for bit; from lengths and from offsets; keys in and out of order."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal
from test_tbe_gpu import DEV, _from_lengths, _launch_text, build

pytestmark = pytest.mark.gpu

SPECS = {
    # lane chunks of 16, 8 and 4 bytes of one type, 1 to 64 lanes a row
    "int8": [(O.INT8, 300, d) for d in (4, 12, 8, 40, 64, 72, 80, 112, 128, 256, 1024)],
    # int4 and int2 rows in the chunks of at most 16 accumulators
    "sub-byte": [(O.INT4, 300, 128), (O.INT4, 310, 256), (O.INT4, 290, 40), (O.INT2, 300, 256), (O.INT2, 320, 16),
                 (O.INT2, 280, 80), (O.INT8, 250, 64)],
    "mixed": [((O.INT8, O.INT4, O.INT2, O.FP16)[t % 4], 200 + t, (32, 64, 128, 256)[t // 4]) for t in range(16)],
    "floats": [(O.FP16, 300, 2), (O.FP16, 300, 20), (O.FP16, 300, 72), (O.FP32, 300, 1), (O.FP32, 300, 6), (O.FP32, 300, 100)],
}


@pytest.mark.parametrize("weights", ["none", "sample", "position"])
@pytest.mark.parametrize("name", list(SPECS))
def test_one_launch_of_several_classes(tuning, name, weights):
    tuning(balanced=1, window=96)
    rng = np.random.default_rng(len(name) * 7 + len(weights))
    specs = SPECS[name]
    T, B = len(specs), 131
    idt, pooling, out = {"none": (np.int32, O.SUM, O.FP16), "sample": (np.int64, O.MEAN, O.FP32),
                         "position": (np.int64, O.SUM, O.FP16)}[weights]
    tbe, store = build(rng, specs, list(range(T)), pooling, out, 16)
    for order in (list(range(T)), list(rng.permutation(T + 1)[:T])):
        K = max(order) + 1
        lengths = rng.choice([0, 1, 3, 4, 5, 8, 9, 40], K * B).astype(idt)
        starts = np.concatenate([[0], np.cumsum(lengths)])
        ids = rng.integers(-1, 200, int(starts[-1])).astype(idt)
        # the oracle takes the features' bags in feature order
        picks = np.concatenate([np.arange(p * B, (p + 1) * B) for p in order])
        seg = np.concatenate([np.arange(starts[q], starts[q + 1]) for q in picks])
        offsets = np.zeros(T * B + 1, dtype=idt)
        offsets[1:] = np.cumsum(lengths[picks])
        psw, kw = None, {}
        if weights == "sample":
            psw = rng.uniform(-1, 1, len(ids)).astype(np.float32)
        elif weights == "position":
            table = rng.uniform(-1, 1, 6 * K).astype(np.float32)
            start, n = [6 * k for k in range(K)], [6 if k % 3 else 0 for k in range(K)]
            key = np.repeat(np.arange(K * B) // B, lengths)
            place = np.arange(len(ids)) - np.repeat(starts[:-1], lengths)
            w = np.where(np.take(n, key) > 0, table[np.take(start, key) + np.minimum(place, 5)], 1.0).astype(np.float32)
            kw = {"position_weights": (torch.from_numpy(table).to(DEV), start, n)}
        full = psw if weights == "sample" else w if weights == "position" else None
        want = O.tbe_forward(store, list(range(T)), B, ids[seg], offsets, None if full is None else full[seg], pooling, out)
        got = _from_lengths(tbe, ids, lengths, psw, B, feature_positions=order, **kw)
        assert bits_equal(got, want) == 0, order
        t_off = torch.from_numpy(starts.astype(idt)).to(DEV)
        got = tbe(torch.from_numpy(ids).to(DEV), t_off, None if psw is None else torch.from_numpy(psw).to(DEV),
                  feature_positions=order, batch_size=B, **kw).cpu().numpy()
        assert bits_equal(got, want) == 0, order
    assert "tbe_pooled_multi_kernel" in _launch_text(tbe, B, len(ids), T)
    assert tbe.out_of_range_count() == 0


def test_route_is_the_same_from_lengths_and_from_offsets():
    """Seven launch classes: one launch below 12,000 ids per compute unit, whatever the bags' bounds come from; a launch
    per class from there on.  Few classes own no second stream and take one launch at any size."""
    rng = np.random.default_rng(21)
    dts, dims = (O.INT8, O.INT4, O.INT2, O.FP16), (32, 64, 128, 256)
    seven, _ = build(rng, [(dts[t % 4], 50, dims[t // 4]) for t in range(16)], list(range(16)), O.SUM, O.FP32, 16)
    two, _ = build(rng, [(dts[t % 2], 50, 64) for t in range(16)], list(range(16)), O.SUM, O.FP32, 16)
    line = 12_000 * torch.cuda.get_device_properties(0).multi_processor_count
    for n_keys in (0, 16):
        assert "tbe_pooled_multi_kernel" in _launch_text(seven, 4096, line - 1, n_keys)
        assert _launch_text(seven, 4096, line, n_keys).count("tbe_pooled_cu_kernel") == 7
        assert "tbe_pooled_multi_kernel" in _launch_text(two, 4096, 2 * line, n_keys)


@pytest.mark.parametrize("name", ["features", "cut row"])
def test_no_one_launch_of_windows(name):
    """Plans of several classes that windows cannot serve in one launch: the sixteen-lane kernel, one launch for all
    classes, up to 2500 ids per compute unit, whatever the number of bags; windows, a launch per class, from there on.
    Few ids in many bags against the oracle."""
    rng = np.random.default_rng(len(name))
    specs = {"features": [((O.INT8, O.FP16)[t % 2], 50 + t, 16) for t in range(130)],
             "cut row": [(O.INT8, 60, 16)] * 15 + [(O.FP32, 40, 1028)]}[name]
    T = len(specs)
    tbe, store = build(rng, specs, list(range(T)), O.SUM, O.FP16, 16)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    B = 80 * cus // T + 1
    lengths = rng.choice([0, 0, 1, 2, 9], T * B).astype(np.int32)
    offsets = np.zeros(T * B + 1, dtype=np.int32)
    offsets[1:] = np.cumsum(lengths)
    ids = rng.integers(0, 40, int(offsets[-1])).astype(np.int32)
    assert len(ids) < 2500 * cus and "tbe_pooled_kernel" in _launch_text(tbe, B, len(ids), T)
    for n_keys in (0, T):
        assert "tbe_pooled_kernel" in _launch_text(tbe, B, 2500 * cus - 1, n_keys)
        assert "tbe_pooled_cu_kernel" in _launch_text(tbe, B, 2500 * cus, n_keys)
    want = O.tbe_forward(store, list(range(T)), B, ids, offsets, None, O.SUM, O.FP16)
    assert bits_equal(_from_lengths(tbe, ids, lengths, None, B), want) == 0
    got = tbe(torch.from_numpy(ids).to(DEV), torch.from_numpy(offsets).to(DEV)).cpu().numpy()
    assert bits_equal(got, want) == 0
