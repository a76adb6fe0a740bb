"""Results of the window kernel: one to sixteen 16-byte vectors per lane, lane groups of every kind, rows that begin off a
16-byte boundary, both result types, SUM and MEAN; against the CPU oracle, bit for bit."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal
from test_tbe_gpu import _from_lengths, build

pytestmark = pytest.mark.gpu


# (lanes behind a wave's last whole group, rows of one lane, results of less than a vector a lane, several slices of a row)
@pytest.mark.parametrize("dtype,dims", [
    (O.INT8, (4, 32, 40, 72, 104, 128, 256, 1040)), (O.INT4, (8, 64, 104, 128, 512)), (O.INT2, (16, 48, 128, 256, 1024)),
    (O.FP16, (2, 32, 36, 104, 512)), (O.FP32, (1, 4, 36, 256)),
])
@pytest.mark.parametrize("out", [O.FP16, O.FP32])
@pytest.mark.parametrize("mode", [O.SUM, O.MEAN])
@pytest.mark.parametrize("window", [0, 70])
def test_results(tuning, dtype, dims, out, mode, window):
    tuning(balanced=1, window=window)
    for dim in dims:
        for first in (dim, 4 if dtype != O.INT2 else 16):  # (the narrow feature in front shifts the others' columns)
            rng = np.random.default_rng([int(dtype), dim, first])
            B = 37
            specs = [(dtype, 60, max(first, 8 if dtype == O.INT4 else first)), (dtype, 50, dim), (dtype, 70, dim)]
            tbe, store = build(rng, specs, [0, 1, 2], mode, out, 16)
            lengths = rng.choice([0, 1, 2, 9], 3 * B).astype(np.int64)
            offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
            ids = rng.integers(-1, 50, int(offsets[-1])).astype(np.int64)
            want = O.tbe_forward(store, [0, 1, 2], B, ids, offsets, None, mode, out)
            assert bits_equal(_from_lengths(tbe, ids, lengths, None, B), want) == 0, (dim, first)
            got = tbe(indices=torch.from_numpy(ids).cuda(), offsets=torch.from_numpy(offsets).cuda()).cpu().numpy()
            assert bits_equal(got, want) == 0, (dim, first)


# Lanes of 32 and 64 accumulators, which look up anew behind the pooling loop where a bag's results go: lane groups of every
# kind (5, 6, 8, 16 and 64 lanes), more features in a window than its descriptors hold, waves of several rounds.
@pytest.mark.parametrize("dtype,dim", [(O.INT4, 160), (O.INT4, 192), (O.INT4, 256), (O.INT4, 512), (O.INT4, 2080),
                                       (O.INT2, 128), (O.INT2, 192), (O.INT2, 320), (O.INT2, 512)])
@pytest.mark.parametrize("F,B", [(3, 211), (45, 5)])
@pytest.mark.parametrize("weighted,idt", [(False, np.int32), (True, np.int64)])
def test_wide_lanes(tuning, dtype, dim, F, B, weighted, idt):
    tuning(balanced=1, window=256)
    rng = np.random.default_rng([int(dtype), dim, F])
    ftm = [f % 2 for f in range(F)]
    for mode, out in ((O.SUM, O.FP16), (O.MEAN, O.FP32)):
        tbe, store = build(rng, [(dtype, 60, dim), (dtype, 50, dim)], ftm, mode, out, 16)
        lengths = rng.choice([0, 1, 3, 8, 17, 40], F * B).astype(idt)
        offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(idt)
        ids = rng.integers(-1, 50, int(offsets[-1])).astype(idt)
        psw = rng.random(len(ids)).astype(np.float32) if weighted else None
        want = O.tbe_forward(store, ftm, B, ids, offsets, psw, mode, out)
        assert bits_equal(_from_lengths(tbe, ids, lengths, psw, B), want) == 0
        got = tbe(torch.from_numpy(ids).cuda(), torch.from_numpy(offsets).cuda(),
                  None if psw is None else torch.from_numpy(psw).cuda()).cpu().numpy()
        assert bits_equal(got, want) == 0


# Blocks of one round to many times what their sixteen waves hold, numbers that leave some SIMDs a round more than others:
# every round is pooled once.
@pytest.mark.parametrize("dtype,dim,per_round", [(O.INT8, 256, 4), (O.INT8, 1024, 1), (O.FP16, 32, 8), (O.INT4, 512, 4)])
@pytest.mark.parametrize("rounds", [1, 15, 16, 17, 18, 19, 20, 21, 33, 47])
def test_every_round_once(tuning, dtype, dim, per_round, rounds):
    tuning(balanced=1, window=rounds * per_round)
    rng = np.random.default_rng([rounds, dim])
    B = rounds * per_round + 3
    tbe, store = build(rng, [(dtype, 60, dim), (dtype, 50, dim)], [0, 1], O.SUM, O.FP32, 16)
    lengths = rng.choice([0, 1, 5, 30], 2 * B).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ids = rng.integers(0, 50, int(offsets[-1])).astype(np.int32)
    want = O.tbe_forward(store, [0, 1], B, ids, offsets, None, O.SUM, O.FP32)
    assert bits_equal(_from_lengths(tbe, ids, lengths, None, B), want) == 0
    # (in place of the next call's results, so that a round left out shows)
    out = torch.full((B, 2 * dim), float("nan"), device="cuda")
    tbe(indices=torch.from_numpy(ids).cuda(), offsets=torch.from_numpy(offsets).cuda(), batch_size=B, out=out)
    assert bits_equal(out.cpu().numpy(), want) == 0
