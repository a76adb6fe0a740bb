"""Sequence lookup from key totals and key starts, and the per-key counts that
feed it, on the GPU against the CPU oracle."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal
from test_tbe_gpu import build
from torchrec_amd import _lib, KeyedJaggedTensor, ops
from torchrec_amd.modules.embedding_configs import DataType, EmbeddingConfig
from torchrec_amd.quant import EmbeddingCollection as QuantEC

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# One lane per row, lanes that are no power of two, rows of 2 and of 4 output vectors per lane, several column slices.
@pytest.mark.parametrize("dtype,dim,out", [(O.INT8, 4, O.FP16), (O.INT8, 36, O.FP16), (O.INT8, 128, O.FP16), (O.INT8, 64, O.FP32),
                                           (O.INT4, 104, O.FP16), (O.INT4, 128, O.FP32), (O.INT2, 64, O.FP16),
                                           (O.FP16, 40, O.FP32), (O.FP32, 8, O.FP16), (O.INT8, 1028, O.FP16)])
# Ids per key: fewer than a tile, exactly tiles, uneven and empty keys, more keys than a wave has lanes.
@pytest.mark.parametrize("totals", [[1], [64, 128, 256, 512], [0, 5000, 0, 3, 129], [7] * 130, [70_000, 1, 2_000]])
@pytest.mark.parametrize("idt", [np.int32, np.int64])
def test_sequence_from_totals_and_starts(dtype, dim, out, totals, idt):
    rng = np.random.default_rng(dim * len(totals))
    K = len(totals)
    if dim > 1000 and sum(totals) > 10_000:
        pytest.skip("wide rows are checked on the short inputs")
    tables = min(K, 5)
    specs = [(dtype, 50 + 31 * t, dim) for t in range(tables)]
    ftm = sorted(f % tables for f in range(K))
    tbe, store = build(rng, specs, ftm, O.NONE, out, 16)
    ids = np.concatenate([rng.integers(-1, specs[ftm[f]][1], n) for f, n in enumerate(totals)]).astype(idt)
    starts = np.concatenate([[0], np.cumsum(totals)])
    want = O.tbe_forward(store, ftm, 1, ids, starts.astype(idt), None, O.NONE, out)
    dids = torch.from_numpy(ids).to(DEV)
    routes = {"totals": {"key_totals": torch.tensor(totals, device=DEV)}, "offsets": {"offsets": torch.from_numpy(starts.astype(idt)).to(DEV)}}
    if K <= 128:
        routes["starts"] = {"key_starts": starts.tolist()}
    for name, kw in routes.items():
        got = tbe(indices=dids, **{"offsets": None, **kw}).cpu().numpy()
        assert bits_equal(got, want) == 0, name
    assert tbe.out_of_range_count() == 0


def test_sequence_features_at_other_positions():
    """Features out of key order, a key no feature sits at, one key that two features share, a padded ids buffer."""
    rng = np.random.default_rng(2)
    tbe, store = build(rng, [(O.INT8, 300, 64), (O.INT4, 200, 64)], [0, 0, 1], O.NONE, O.FP16, 16)
    totals = [300, 0, 170, 40]
    starts = np.concatenate([[0], np.cumsum(totals)])
    ids = rng.integers(0, 200, 510).astype(np.int64)
    padded = torch.from_numpy(np.concatenate([ids, np.full(9, 10**6)])).to(DEV)
    out = torch.full((519, 64), 7.0, dtype=torch.float16, device=DEV)
    for positions in ([2, 0, 3], [2, 2, 0]):
        for kw in ({"key_totals": torch.tensor(totals, device=DEV)}, {"key_starts": starts.tolist()}):
            out.fill_(7.0)
            tbe(indices=padded, offsets=None, feature_positions=positions, out=out, **kw)
            got = out.cpu().numpy()
            seen = np.zeros(519, bool)
            for f, p in enumerate(positions):
                if positions.count(p) > 1:
                    seen[starts[p]:starts[p + 1]] = True  # two features write here: either may stand
                    continue
                part = ids[starts[p]:starts[p + 1]]
                one = O.tbe_forward(store, [0, 0, 1], 1, np.concatenate([part] * 3),
                                    np.arange(4) * len(part), None, O.NONE, O.FP16)
                assert bits_equal(got[starts[p]:starts[p + 1]], one[f * len(part):(f + 1) * len(part)]) == 0
                seen[starts[p]:starts[p + 1]] = True
            assert (got[~seen] == 7.0).all()
    assert tbe.out_of_range_count() == 0


@pytest.mark.parametrize("K,B", [(1, 1), (1, 5000), (3, 7), (26, 2048), (256, 3), (257, 3), (1024, 2), (1025, 2)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("skip", [0, 1])  # 1: the lengths start off a 16-byte boundary
def test_key_totals(K, B, dtype, skip):
    lengths = torch.randint(0, 50, (K * B + skip,), dtype=dtype, device=DEV)[skip:]
    want = lengths.view(K, B).sum(1).tolist()
    assert ops.length_per_key(lengths, K, B) == want
    offsets = ops.asynchronous_complete_cumsum(lengths)
    for bags, are_offsets in ((lengths, False), (offsets, True)):
        begun = ops.key_totals_begin(bags, are_offsets, K, B, on_device=True)
        assert (begun is None) == (K > 1024)
        if begun is not None:
            totals, finish = begun
            assert finish() == want and totals.tolist() == want


def test_key_totals_threads_and_open_calls():
    """More calls open than there are slots (the surplus takes the copying route), and threads on streams of their own."""
    lengths = [torch.full((6,), i, dtype=torch.int32, device=DEV) for i in range(80)]
    later = [ops.length_per_key_async(t, 2, 3) for t in lengths]
    assert [f() for f in later] == [[3 * i, 3 * i] for i in range(80)]
    bad = []

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            for i in range(50):
                t = torch.full((4 * 33,), seed * 50 + i, dtype=torch.int64, device=DEV)
                if ops.length_per_key(t, 4, 33) != [33 * (seed * 50 + i)] * 4:
                    bad.append((seed, i))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_key_totals_after_an_earlier_error():
    """An error that another HIP call left behind is reported with nothing queued: a kernel under way would store its
    totals into a slot that was given back, and that the next call may hold."""
    l, hip = _lib.lib(), ctypes.CDLL(_lib.LIB_PATH)  # (the HIP runtime this library is linked to)
    lengths, totals = torch.arange(12, device=DEV), torch.full((3,), -7, device=DEV)
    ticket = ctypes.c_int32(5)
    args = (lengths.data_ptr(), 0, 3, 4, 1, totals.data_ptr(), ctypes.byref(ticket), _lib.current_stream(DEV))
    torch.cuda.synchronize()
    assert hip.hipSetDevice(1 << 20) != 0
    assert l.tra_key_totals_begin(*args) != 0 and b"earlier" in l.tra_last_error() and ticket.value == -1
    torch.cuda.synchronize()
    assert totals.tolist() == [-7] * 3
    assert l.tra_key_totals_begin(*args) == 0
    host = (ctypes.c_int64 * 3)()
    assert l.tra_key_totals_wait(ticket, host) == 0
    assert list(host) == totals.tolist() == [6, 22, 38]


def test_key_totals_reject_other_integer_types():
    with pytest.raises(TypeError):
        ops.length_per_key(torch.ones(4, dtype=torch.int16, device=DEV), 2, 2)


@pytest.mark.parametrize("K,dim", [(64, 1024), (65, 1024), (128, 8), (129, 8)])
def test_collection_of_more_slices_than_key_starts(K, dim):
    """One feature more than the launch arguments hold key starts of, in rows of one and of two column slices, from a
    KJT without its per-key counts and with them (which the first call leaves on it)."""
    rng = np.random.default_rng(K)
    rows = torch.randn(9, dim, device=DEV).half()
    config = EmbeddingConfig(name="t", embedding_dim=dim, num_embeddings=9, feature_names=[f"f{k}" for k in range(K)],
                             data_type=DataType.FP16)
    qec = QuantEC([config], DEV, output_dtype=torch.half,
                  table_name_to_quantized_weights={"t": (rows.view(torch.uint8), None)})
    assert qec._emb_modules[0].takes_key_starts() == (K * (2 if dim == 1024 else 1) <= 128)
    lengths = torch.from_numpy(rng.integers(0, 4, 3 * K)).to(DEV)
    ids = torch.from_numpy(rng.integers(0, 9, int(lengths.sum()))).to(DEV)
    kjt = KeyedJaggedTensor(keys=[f"f{k}" for k in range(K)], values=ids, lengths=lengths)
    for _ in range(2):
        got = qec(kjt)
        assert torch.equal(torch.cat([got[k].values() for k in kjt.keys()]), rows[ids])
        assert kjt.length_per_key_or_none() is not None


def test_collection_saved_without_its_flat_names():
    """A collection that was saved before it kept its embedding names in one list."""
    tables = [EmbeddingConfig(name=f"t{k}", embedding_dim=8, num_embeddings=9, feature_names=[f"f{k}"],
                              data_type=DataType.INT8 if k else DataType.FP16) for k in range(2)]
    qec = QuantEC(tables, DEV, output_dtype=torch.half)
    kjt = KeyedJaggedTensor(keys=["f1", "f0"], values=torch.tensor([1, 2, 3], device=DEV), lengths=torch.tensor([1, 2], device=DEV))
    want = qec(kjt)
    qec.__dict__.pop("_flat_embedding_names")
    got = qec(kjt)
    assert list(got) == list(want) and all(torch.equal(got[k].values(), want[k].values()) for k in want)
