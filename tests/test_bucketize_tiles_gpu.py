"""Bucketization by four launches and by two at the sizes where its tiles, steps of ids and bitmap words
begin and end, against the oracle: whole numbers, compared exactly."""
import numpy as np
import pytest
import torch

import oracle as O
from torchrec_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lengths(how, n, rng):
    if how == "even":
        return rng.integers(0, 9, n)
    lengths = np.zeros(n, dtype=np.int64)
    if how == "words":  # bags that end on, in front of and behind a wave's 64 ids, with empty ones between
        lengths[::2] = rng.choice([1, 63, 64, 65, 127, 128], len(lengths[::2]))
    elif how == "long":  # bags of several steps beside empty ones
        lengths[rng.integers(0, n, 3)] = [4095, 4097, 9000]
        lengths[n - 1] = 1
    return lengths


@pytest.mark.parametrize("F,B,W,how", [
    (5, 3277, 3, "even"),     # 16385 lengths: the first count whose bounds come from launches of their own
    (4, 4096, 3, "even"),     # 16384: the last that takes two
    (70, 300, 5, "even"),     # some hundred tiles
    (300, 80, 64, "even"),    # the most buckets
    (1, 20000, 1, "even"),    # one bucket
    (3, 6000, 7, "words"),
    (2, 700, 8, "words"),     # two launches
    (2, 9001, 4, "long"),
    (3, 50, 33, "long"),
])
@pytest.mark.parametrize("idt", [np.int32, np.int64])
def test_tiles(F, B, W, how, idt):
    rng = np.random.default_rng(F * 1000 + B + W)
    lengths = _lengths(how, F * B, rng).astype(idt)
    # block sizes from one row to 2^30, one of them beyond 32 bits where the ids can be
    block_sizes = (2 ** rng.uniform(0, 30, F)).astype(np.int64)
    if idt == np.int64:
        block_sizes[0] = 3 * 2**33
    per_key = lengths.reshape(F, B).sum(1)
    top = np.iinfo(idt).max
    ids = np.concatenate([rng.integers(0, min(int(bs) * (W + 1), top), n) for bs, n in zip(block_sizes, per_key)])
    ids[rng.random(len(ids)) < 0.001] = top  # (beyond the last bucket, and in no 32-bit wave)
    ids = ids.astype(idt)
    weights = rng.random(len(ids)).astype(np.float32)
    nl, ni, nw, nu = O.bucketize(lengths, ids, block_sizes, W, weights, False, return_permute=True)
    gl, gi, gw, _, gu = ops.block_bucketize_sparse_features(
        torch.from_numpy(lengths).to(DEV), torch.from_numpy(ids).to(DEV), False, True,
        torch.from_numpy(block_sizes).to(DEV), W, torch.from_numpy(weights).to(DEV), False)
    assert np.array_equal(gl.cpu().numpy(), nl)
    assert np.array_equal(gi.cpu().numpy(), ni)
    assert np.array_equal(gw.cpu().numpy(), nw)
    assert np.array_equal(gu.cpu().numpy(), nu)


# Ids, weights and places of more than 256 MB, whose blocks share a compute unit with fewer others, and of a little less.
@pytest.mark.parametrize("mean", [3190, 3205])
def test_more_than_the_cache_holds(mean):
    rng = np.random.default_rng(mean)
    F, B, W = 3, 700, 3
    lengths = rng.integers(mean - 5, mean + 6, F * B)
    n = int(lengths.sum())
    assert (40 * n > 2**28) == (mean > 3200)
    ids = rng.integers(0, 1000, n)
    weights = rng.random(n).astype(np.float32)
    block_sizes = np.full(F, 334)
    nl, ni, nw, nu = O.bucketize(lengths, ids, block_sizes, W, weights, False, return_permute=True)
    gl, gi, gw, _, gu, gb = ops._block_bucketize(
        torch.from_numpy(lengths).to(DEV), torch.from_numpy(ids).to(DEV), False, True,
        torch.from_numpy(block_sizes).to(DEV), W, torch.from_numpy(weights).to(DEV), False, want_buckets=True)
    for got, want in ((gl, nl), (gi, ni), (gw, nw), (gu, nu), (gb, ids // 334)):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("F,B", [(3, 100), (40, 700)])
@pytest.mark.parametrize("bad", [-1, 10**6])
def test_lengths_that_are_no_partition(F, B, bad):
    """Found by the first launch, whichever tile holds it: the same as bags written out one after the other."""
    rng = np.random.default_rng(B)
    lengths = rng.integers(0, 9, F * B)
    ids = rng.integers(0, 1000, int(lengths.sum()))
    at = F * B // 2
    good = torch.from_numpy(lengths).to(DEV)
    lengths[at] = bad
    args = (torch.from_numpy(ids).to(DEV), False, False, torch.full((F,), 300, dtype=torch.int64, device=DEV), 4)
    nl, ni, _, _, _ = ops.block_bucketize_sparse_features(torch.from_numpy(lengths).to(DEV), *args)
    offsets = np.clip(np.concatenate([[0], np.cumsum(lengths)]), 0, len(ids))
    sizes = np.maximum(offsets[1:] - offsets[:-1], 0)
    moved = np.concatenate([ids[s:s + n] for s, n in zip(offsets[:-1], sizes)])
    want = O.bucketize(sizes, moved, np.full(F, 300), 4, None, False)
    assert np.array_equal(nl.cpu().numpy(), want[0]) and np.array_equal(ni.cpu().numpy(), want[1])
    # and the call after it is none the wiser
    nl, ni, _, _, _ = ops.block_bucketize_sparse_features(good, *args)
    want = O.bucketize(good.cpu().numpy(), ids, np.full(F, 300), 4, None, False)
    assert np.array_equal(nl.cpu().numpy(), want[0]) and np.array_equal(ni.cpu().numpy(), want[1])
