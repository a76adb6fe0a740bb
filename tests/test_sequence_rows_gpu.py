"""The row ranges that a sequence collection hands out, against lookups of one key at a time."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal
from test_tbe_gpu import build
from torchrec_amd import KeyedJaggedTensor
from torchrec_amd.modules.embedding_configs import DataType, EmbeddingConfig
from torchrec_amd.quant import EmbeddingCollection as QuantEC

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _collection(features, need_indices=False):
    tables = [EmbeddingConfig(name="t%d" % i, embedding_dim=16, num_embeddings=97, feature_names=["f%d" % i],
                              data_type=DataType.INT8) for i in range(features)]
    module = QuantEC(tables, DEV, need_indices=need_indices, output_dtype=torch.float)
    for op in module._emb_modules:
        for payload, scale, bias in op.split_embedding_weights_with_scale_bias(2):
            payload.view(torch.int32).random_(-(2**31), 2**31 - 1)
            scale.uniform_(0.01, 0.02)
            bias.uniform_(-1, 0)
    return module


# Ids per bag of each key; the collection's features among the keys (half of them and more: all ranges at once; fewer:
# one by one), empty keys in front, between and behind, ids behind the last bag's, a negative length.
@pytest.mark.parametrize("bags,used,tail", [
    ([[1, 2]], [0], 0), ([[0, 0], [3, 1], [0, 0]], [0, 1, 2], 0), ([[4, 1], [0, 0], [2, 2], [1, 0]], [3, 0], 3),
    ([[4, 1], [0, 5], [2, 2], [1, 0], [1, 1]], [2, 1], 2), ([[2, 1], [3, -1], [2, 2]], [0, 1, 2], 4),
    ([[2, 1], [-4, 1], [2, 2]], [0, 1, 2], 9), ([[0, 0], [0, 0]], [1, 0], 1),
])
@pytest.mark.parametrize("counts_known", [False, True])
@pytest.mark.parametrize("need_indices", [False, True])
def test_row_ranges(bags, used, tail, counts_known, need_indices):
    keys = [None] * len(bags)
    for f, k in enumerate(used):
        keys[k] = "f%d" % f
    keys = [k or "unused%d" % i for i, k in enumerate(keys)]
    module = _collection(len(used), need_indices)
    per_key = [sum(b) for b in bags]
    starts = np.concatenate([[0], np.cumsum(per_key)])
    n = max(int(starts.max()), 0) + tail
    ids = torch.randint(0, 97, (n,), device=DEV)
    lengths = torch.tensor(sum(bags, []), device=DEV)
    kjt = KeyedJaggedTensor(keys=keys, values=ids, lengths=lengths, length_per_key=per_key if counts_known else None)
    out = module(kjt)
    assert list(out) == ["f%d" % f for f in range(len(used))]
    for f, k in enumerate(used):
        jt = out["f%d" % f]
        mine = ids[starts[k] : starts[k + 1]]
        assert jt.values().shape == (mine.numel(), 16) and jt.values().is_contiguous()
        assert jt.lengths().tolist() == bags[k]
        if min(b for key in bags for b in key) >= 0:  # (else: which of the overlapping keys' rows are written is not said)
            one = KeyedJaggedTensor(keys=["f%d" % i for i in range(len(used))], values=mine,
                                    lengths=torch.tensor([mine.numel() if i == f else 0 for i in range(len(used))], device=DEV))
            assert torch.equal(jt.values(), module(one)["f%d" % f].values())
        assert (torch.equal(jt.weights(), mine)) if need_indices else jt.weights_or_none() is None


# One to sixteen 16-byte vectors of results per lane, rows that are and are not multiples of 16 bytes or of a line, lane
# groups that leave lanes of the wave idle, a row in several column slices; tiles that begin at any row and end inside a
# wave's step.
@pytest.mark.parametrize("dtype,dims", [
    (O.INT8, (4, 12, 32, 40, 72, 96, 104, 128, 192, 256, 1040)), (O.INT4, (8, 40, 64, 104, 128, 256, 512)),
    (O.INT2, (16, 48, 64, 128, 256, 1024)), (O.FP16, (2, 8, 32, 36, 104, 128, 512)), (O.FP32, (1, 4, 36, 128, 256)),
])
@pytest.mark.parametrize("out", [O.FP16, O.FP32])
def test_results_of_all_widths(dtype, dims, out):
    rng = np.random.default_rng(int(dtype))
    for dim in dims:
        totals = [3, 0, 61, 1, 700, 5]
        specs = [(dtype, 40 + 7 * t, dim) for t in range(3)]
        ftm = [0, 0, 1, 1, 2, 2]
        tbe, store = build(rng, specs, ftm, O.NONE, out, 16)
        ids = np.concatenate([rng.integers(-1, specs[ftm[f]][1], n) for f, n in enumerate(totals)]).astype(np.int64)
        starts = np.concatenate([[0], np.cumsum(totals)])
        want = O.tbe_forward(store, ftm, 1, ids, starts, None, O.NONE, out)
        guard = torch.full((ids.size + 40, dim), 7.0, dtype=torch.half if out == O.FP16 else torch.float, device=DEV)
        tbe(indices=torch.from_numpy(ids).to(DEV), offsets=None, key_starts=starts.tolist(), out=guard)
        got = guard.cpu().numpy()
        assert bits_equal(got[: ids.size], want) == 0, dim
        assert (got[ids.size :] == 7.0).all(), dim


# Ids enough for tiles of several rows a lane group (4 steps of `rows` rows); features that end at every place of a tile's
# steps: in front of a wave's first row, inside its rows, behind them.
@pytest.mark.parametrize("dtype,dim,rows", [(O.INT8, 1024, 4), (O.FP16, 512, 4), (O.INT4, 1024, 8), (O.INT8, 512, 4)])
@pytest.mark.parametrize("out", [O.FP16, O.FP32])
def test_steps_that_a_tile_does_not_fill(dtype, dim, rows, out):
    rng = np.random.default_rng(dim + rows)
    step = 4 * rows
    totals = [step + 1, 0, 3, 2 * step - 1, rows, rows + 1, 3 * rows - 1, step]
    totals.append(512 * step)
    specs = [(dtype, 300, dim)]
    ftm = [0] * len(totals)
    tbe, store = build(rng, specs, ftm, O.NONE, out, 16)
    ids = rng.integers(-1, 301, sum(totals)).astype(np.int32)
    starts = np.concatenate([[0], np.cumsum(totals)]).astype(np.int32)
    want = O.tbe_forward(store, ftm, 1, np.where(ids == 300, np.int32(-1), ids), starts, None, O.NONE, out)
    guard = torch.full((ids.size + 40, dim), 7.0, dtype=torch.half if out == O.FP16 else torch.float, device=DEV)
    tbe(indices=torch.from_numpy(ids).to(DEV), offsets=None, key_starts=starts.tolist(), out=guard)
    got = guard.cpu().numpy()
    assert bits_equal(got[: ids.size], want) == 0
    assert (got[ids.size :] == 7.0).all()
    # (ids outside the table are counted once a row, also in steps that are cut short)
    assert tbe.out_of_range_count() == int((ids == 300).sum())


def test_row_ranges_of_given_key_offsets():
    module = _collection(2)
    ids = torch.arange(8, device=DEV)
    kjt = KeyedJaggedTensor(keys=["f0", "f1"], values=ids, lengths=torch.tensor([2, 1, 4, 1], device=DEV),
                            offset_per_key=[0, 3, 8])
    out = module(kjt)
    assert [out[k].values().shape[0] for k in ("f0", "f1")] == [3, 5]
    assert kjt.length_per_key_or_none() is None  # (nothing was added up for it)


def test_rows_may_be_changed_in_place_with_a_gradient():
    module = _collection(3)
    kjt = KeyedJaggedTensor(keys=["f0", "f1", "f2"], values=torch.arange(9, device=DEV),
                            lengths=torch.tensor([1, 2, 3, 0, 2, 1], device=DEV))
    out = module(kjt)
    before = out["f1"].values().clone()
    scale = torch.full((1,), 2.0, device=DEV, requires_grad=True)
    out["f1"].values().mul_(scale).sum().backward()
    assert torch.allclose(scale.grad, before.sum())
    assert not out["f0"].values().requires_grad
