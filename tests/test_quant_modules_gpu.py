"""QuantEmbeddingBagCollection / QuantEmbeddingCollection end to end on the GPU:
from_float, key order, shared features, weighted, state_dict round trip.
Numerics are compared with the CPU oracle fed by the module's own packed store
(bit-exact), and with the float module at the reference's own loose tolerance
(atol 0.1, torchrec/quant/tests/test_embedding_modules.py:126)."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal
from torchrec_amd import KeyedJaggedTensor
from torchrec_amd.modules.embedding_configs import DataType, EmbeddingBagConfig, EmbeddingConfig, PoolingType, QuantConfig
from torchrec_amd.modules.embedding_modules import EmbeddingBagCollection, EmbeddingCollection
from torchrec_amd.quant.embedding_modules import (
    _fx_trec_unwrap_kjt,
    EmbeddingBagCollection as QuantEBC,
    EmbeddingCollection as QuantEC,
    quant_prep_enable_quant_state_dict_split_scale_bias,
    quantize_state_dict,
)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
OCODE = {"fp32": O.FP32, "fp16": O.FP16, "int8": O.INT8, "int4": O.INT4, "int2": O.INT2}


def oracle_store_of(tbe):
    """The oracle's view of a module's packed buffer (same bytes, read back from HBM)."""
    return O.Store(
        tbe.weights_dev.cpu().numpy(),
        np.asarray(tbe.weights_physical_offsets, dtype=np.int64),
        np.asarray(tbe.rows, dtype=np.int64),
        np.asarray(tbe.dims, dtype=np.int32),
        np.asarray([OCODE[str(t)] for t in tbe.weight_tys], dtype=np.int32),
        np.asarray(tbe.row_stride, dtype=np.int32),
    )


def qconfig(weight_dtype, out_dtype, per_table=None):
    act = torch.quantization.PlaceholderObserver.with_args(dtype=out_dtype)
    w = torch.quantization.PlaceholderObserver.with_args(dtype=weight_dtype)
    return QuantConfig(activation=act, weight=w, per_table_weight_dtype=per_table) if per_table else torch.quantization.QConfig(activation=act, weight=w)


def random_kjt(rng, keys, rows, B, max_len, weighted=False, idt=torch.int64):
    F = len(keys)
    lengths = rng.integers(0, max_len + 1, F * B)
    per = lengths.reshape(F, B).sum(axis=1)
    ids = np.concatenate([rng.integers(0, rows[f], per[f]) for f in range(F)])
    return KeyedJaggedTensor(
        keys=list(keys), values=torch.from_numpy(ids).to(idt).to(DEV),
        lengths=torch.from_numpy(lengths).to(torch.int32).to(DEV),
        weights=torch.from_numpy(rng.random(len(ids)).astype(np.float32)).to(DEV) if weighted else None)


@pytest.mark.parametrize("weight_dtype", [torch.qint8, torch.quint4x2, torch.quint2x4, torch.half])
@pytest.mark.parametrize("out_dtype", [torch.float, torch.half])
@pytest.mark.parametrize("weighted", [False, True])
def test_qebc_from_float(weight_dtype, out_dtype, weighted):
    rng = np.random.default_rng(0)
    torch.manual_seed(0)
    tables = [
        EmbeddingBagConfig(name="t1", embedding_dim=16, num_embeddings=10, feature_names=["f1"]),
        # (nn.EmbeddingBag, the float side, has no weighted mean)
        EmbeddingBagConfig(name="t2", embedding_dim=32, num_embeddings=20, feature_names=["f2", "f3"],
                           pooling=PoolingType.SUM if weighted else PoolingType.MEAN),
        EmbeddingBagConfig(name="t3", embedding_dim=64, num_embeddings=30, feature_names=["f1"]),
    ]
    ebc = EmbeddingBagCollection(tables=tables, is_weighted=weighted, device=DEV)
    # KJT key order differs from the module's grouped order and has an unused key
    kjt = random_kjt(rng, ["f3", "unused", "f1", "f2"], [20, 5, 10, 20], B=9, max_len=5, weighted=weighted)
    want_float = ebc(kjt)
    ebc.qconfig = qconfig(weight_dtype, out_dtype)
    qebc = QuantEBC.from_float(ebc)
    got = qebc(kjt)
    assert got.values().dtype == out_dtype and got.values().device == DEV
    if weighted:  # one SUM group, table order kept
        assert got.keys() == ["f1@t1", "f2", "f3", "f1@t3"]
        assert got.length_per_key() == [16, 32, 32, 64]
    else:  # grouped order: SUM tables first (t1, t3), then MEAN (t2)
        assert got.keys() == ["f1@t1", "f1@t3", "f2", "f3"]
        assert got.length_per_key() == [16, 64, 32, 32]
    fl = want_float.to_dict()
    # 0.1 is the reference's own bound for int8/int4; 2-bit rows are coarser
    # (step = range / 3), so their bound against the float module is wider.
    atol = 0.6 if weight_dtype == torch.quint2x4 else 0.1
    for k, v in got.to_dict().items():
        torch.testing.assert_close(v.float(), fl[k].float(), atol=atol, rtol=0)
    # oracle on the module's own packed bytes, group by group
    order = [kjt.keys().index(k) for k in qebc._feature_names]
    perm = kjt.permute(order)
    ids, offs = perm.values().cpu().numpy(), perm.offsets().cpu().numpy().astype(np.int64)
    psw = perm.weights().cpu().numpy() if weighted else None
    B = kjt.stride()
    col, f0 = 0, 0
    gv = got.values().cpu().numpy()
    for tbe, nf in zip(qebc._emb_modules, qebc._feature_splits):
        o = offs[f0 * B:(f0 + nf) * B + 1]
        sl = slice(int(o[0]), int(o[-1]))
        want = O.tbe_forward(oracle_store_of(tbe), tbe.feature_table_map, B, ids[sl], o - o[0],
                             None if psw is None else psw[sl], int(tbe.pooling_mode),
                             O.FP16 if out_dtype == torch.half else O.FP32)
        assert bits_equal(np.ascontiguousarray(gv[:, col:col + tbe.total_D]), want) == 0
        col += tbe.total_D
        f0 += nf


def test_qebc_per_table_dtype_and_int32_ids():
    rng = np.random.default_rng(1)
    tables = [EmbeddingBagConfig(name=f"t{i}", embedding_dim=d, num_embeddings=50, feature_names=[f"f{i}"])
              for i, d in enumerate([32, 64, 128, 256])]
    ebc = EmbeddingBagCollection(tables=tables, device=DEV)
    ebc.qconfig = qconfig(torch.qint8, torch.half, per_table={"t1": torch.quint4x2, "t2": torch.quint2x4, "t3": torch.half})
    qebc = QuantEBC.from_float(ebc)
    assert [str(t) for t in qebc._emb_modules[0].weight_tys] == ["int8", "int4", "int2", "fp16"]
    assert len(qebc._emb_modules) == 1  # one group although dtypes and dims differ
    kjt = random_kjt(rng, ["f0", "f1", "f2", "f3"], [50] * 4, B=33, max_len=12, idt=torch.int32)
    got = qebc(kjt).values().cpu().numpy()
    tbe = qebc._emb_modules[0]
    want = O.tbe_forward(oracle_store_of(tbe), [0, 1, 2, 3], 33, kjt.values().cpu().numpy(),
                         kjt.offsets().cpu().numpy(), None, O.SUM, O.FP16)
    assert bits_equal(got, want) == 0


def test_qebc_state_dict_round_trip():
    torch.manual_seed(3)
    mk = lambda: [EmbeddingBagConfig(name="t1", embedding_dim=16, num_embeddings=10, feature_names=["f1"]),
                  EmbeddingBagConfig(name="t2", embedding_dim=16, num_embeddings=10, feature_names=["f2"])]
    for wd in (torch.qint8, torch.quint4x2, torch.quint2x4):
        for split in (False, True):
            a = EmbeddingBagCollection(tables=mk(), device=DEV)
            b = EmbeddingBagCollection(tables=mk(), device=DEV)
            for m in (a, b):
                m.qconfig = qconfig(wd, torch.float)
                if split:
                    quant_prep_enable_quant_state_dict_split_scale_bias(m)
            qa, qb = QuantEBC.from_float(a), QuantEBC.from_float(b)
            kjt = KeyedJaggedTensor(keys=["f1", "f2"], values=torch.tensor([0, 1, 5, 7], device=DEV),
                                    lengths=torch.tensor([1, 1, 2, 0], device=DEV))
            assert not torch.equal(qa(kjt).values(), qb(kjt).values())
            sd = qa.state_dict()
            assert set(a.state_dict().keys()) <= set(sd.keys())
            qb.load_state_dict(sd)
            for k, v in qb.state_dict().items():
                assert torch.equal(v.view(torch.uint8) if v.dtype == torch.uint8 else v,
                                   sd[k].view(torch.uint8) if v.dtype == torch.uint8 else sd[k])
            assert torch.equal(qa(kjt).values(), qb(kjt).values())


@pytest.mark.parametrize("weight_dtype", [torch.qint8, torch.quint4x2, torch.half])
@pytest.mark.parametrize("need_indices", [False, True])
def test_qec_from_float(weight_dtype, need_indices):
    rng = np.random.default_rng(2)
    tables = [EmbeddingConfig(name="t1", embedding_dim=32, num_embeddings=10, feature_names=["f1", "f2"]),
              EmbeddingConfig(name="t2", embedding_dim=32, num_embeddings=20, feature_names=["f3"])]
    ec = EmbeddingCollection(tables=tables, device=DEV, need_indices=need_indices)
    kjt = random_kjt(rng, ["f3", "f1", "x", "f2"], [20, 10, 4, 10], B=7, max_len=6)
    want_float = ec(kjt)
    ec.qconfig = qconfig(weight_dtype, torch.half, per_table={"t2": torch.quint4x2} if weight_dtype == torch.qint8 else None)
    qec = QuantEC.from_float(ec)
    got = qec(kjt)
    assert set(got.keys()) == {"f1", "f2", "f3"}
    jd = kjt.to_dict()
    for name, jt in got.items():
        assert jt.values().dtype == torch.half
        assert torch.equal(jt.lengths(), jd[name].lengths())
        torch.testing.assert_close(jt.values().float(), want_float[name].values().float(), atol=0.1, rtol=0)
        if need_indices:
            assert torch.equal(jt.weights(), jd[name].values())
        else:
            assert jt.weights_or_none() is None
    # oracle, feature by feature
    f = 0
    for tbe, nf in zip(qec._emb_modules, qec._feature_splits):
        store = oracle_store_of(tbe)
        for k in range(nf):
            name = qec._feature_names[f]
            ids = jd[name].values().cpu().numpy()
            offs = np.array([0, len(ids)], dtype=np.int64)
            t = tbe.feature_table_map[k]
            want = O.tbe_forward(store, [t], 1, ids, offs, None, O.NONE, O.FP16)
            assert bits_equal(got[name].values().cpu().numpy(), want) == 0
            f += 1


def test_qec_shared_feature():
    rng = np.random.default_rng(8)
    tables = [EmbeddingConfig(name="t1", embedding_dim=16, num_embeddings=10, feature_names=["f1"]),
              EmbeddingConfig(name="t2", embedding_dim=16, num_embeddings=10, feature_names=["f1", "f2"])]
    ec = EmbeddingCollection(tables=tables, device=DEV)
    ec.qconfig = qconfig(torch.qint8, torch.float)
    qec = QuantEC.from_float(ec)
    kjt = random_kjt(rng, ["f1", "f2"], [10, 10], B=5, max_len=4)
    got = qec(kjt)
    want = ec(kjt)
    assert set(got.keys()) == {"f1@t1", "f1@t2", "f2"}
    for k in got:
        torch.testing.assert_close(got[k].values(), want[k].values(), atol=0.1, rtol=0)
        assert torch.equal(got[k].lengths(), want[k].lengths())


def test_unwrap_kjt_dtype_rule_device():
    kjt = KeyedJaggedTensor(keys=["a"], values=torch.tensor([1, 2], device=DEV), lengths=torch.tensor([2], device=DEV))
    i, o = _fx_trec_unwrap_kjt(kjt)
    assert i.dtype == torch.int32 and o.dtype == torch.int32


def test_empty_batch_and_empty_features():
    tables = [EmbeddingBagConfig(name="t", embedding_dim=16, num_embeddings=10, feature_names=["f"], data_type=DataType.INT8)]
    q = QuantEBC(tables, False, DEV, output_dtype=torch.half)
    kjt = KeyedJaggedTensor(keys=["f"], values=torch.zeros(0, dtype=torch.int64, device=DEV),
                            lengths=torch.zeros(4, dtype=torch.int32, device=DEV))
    out = q(kjt).values()
    assert out.shape == (4, 16) and not out.any()


def test_qebc_kjt_from_lengths_equals_from_offsets():
    """A KJT built from lengths (the operator derives the offsets) and the same
    KJT built from offsets give identical KeyedTensors."""
    import numpy as np
    from torchrec_amd import KeyedJaggedTensor
    from torchrec_amd.modules.embedding_configs import DataType, EmbeddingBagConfig, PoolingType
    from torchrec_amd.quant import EmbeddingBagCollection as QuantEBC

    dev = torch.device("cuda:0")
    torch.manual_seed(3)
    T, B = 5, 64
    tables = [EmbeddingBagConfig(name=f"t{t}", embedding_dim=32, num_embeddings=500 + t, feature_names=[f"f{t}"],
                                 data_type=DataType.INT4, pooling=PoolingType.SUM) for t in range(T)]
    m = QuantEBC(tables, False, dev, output_dtype=torch.float)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, device=dev))
        for t in range(len(tbe.rows)):  # finite fp16 scale/bias headers
            v = tbe._rows_view(t)
            v[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=dev)
    lengths = torch.randint(0, 9, (T * B,), dtype=torch.int32, device=dev)
    values = torch.randint(0, 500, (int(lengths.sum()),), dtype=torch.int32, device=dev)
    keys = [f"f{t}" for t in range(T)]
    a = m(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths))
    offsets = torch.zeros(T * B + 1, dtype=torch.int32, device=dev)
    offsets[1:] = torch.cumsum(lengths, 0)
    b = m(KeyedJaggedTensor(keys=keys, values=values, offsets=offsets))
    assert a.keys() == b.keys() and torch.equal(a.values(), b.values())
    assert torch.isfinite(a.values()).all()


def test_qebc_short_host_route_and_what_falls_back():
    """forward() takes a short route for the common serving call (one unweighted
    operator, KJT from lengths, keys in module order, contiguous device tensors
    of one integer type).  Its result, and the result of every input that must
    not take it (other key order, a superset of keys, lengths of another integer
    type, non-contiguous ids, a KJT that already holds offsets, the
    cache-features-order flag), against the general route fed with offsets."""
    torch.manual_seed(11)
    T, B = 4, 50
    tables = [EmbeddingBagConfig(name=f"t{t}", embedding_dim=64, num_embeddings=300 + t, feature_names=[f"f{t}"],
                                 data_type=DataType.INT8, pooling=PoolingType.MEAN if t % 2 else PoolingType.SUM)
              for t in range(T)]
    # one pooling type per module so that it is a single operator
    tables = [EmbeddingBagConfig(name=c.name, embedding_dim=c.embedding_dim, num_embeddings=c.num_embeddings,
                                 feature_names=c.feature_names, data_type=c.data_type, pooling=PoolingType.SUM)
              for c in tables]
    m = QuantEBC(tables, False, DEV, output_dtype=torch.half)
    assert len(m._emb_modules) == 1
    tbe = m._emb_modules[0]
    tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, device=DEV))
    for t in range(T):
        tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    keys = [f"f{t}" for t in range(T)]
    lengths = torch.randint(0, 7, (T * B,), dtype=torch.int64, device=DEV)
    values = torch.randint(0, 300, (int(lengths.sum()),), dtype=torch.int64, device=DEV)
    offsets = torch.zeros(T * B + 1, dtype=torch.int64, device=DEV)
    offsets[1:] = torch.cumsum(lengths, 0)
    want = m(KeyedJaggedTensor(keys=keys, values=values, offsets=offsets)).values()

    def same(kjt, module=m):
        got = module(kjt)
        assert got.keys() == keys
        assert torch.equal(got.values().view(torch.int16), want.view(torch.int16))

    same(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths))            # the short route
    same(KeyedJaggedTensor(keys=list(keys), values=values, lengths=lengths))      # an equal list, not the same object
    same(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths.to(torch.int32)))  # lengths of another type
    wide = torch.stack([values, values + 1], dim=1)
    assert not wide[:, 0].is_contiguous()
    same(KeyedJaggedTensor(keys=keys, values=wide[:, 0], lengths=lengths))        # strided ids
    kjt = KeyedJaggedTensor(keys=keys, values=values, lengths=lengths)
    kjt.offsets()                                                                 # offsets already derived
    same(kjt)
    # other key order, and a superset of the keys
    perm = [2, 0, 3, 1]
    Lm = lengths.view(T, B)
    seg = [values[offsets[t * B]:offsets[(t + 1) * B]] for t in range(T)]
    extra = torch.randint(0, 5, (B,), dtype=torch.int64, device=DEV)
    same(KeyedJaggedTensor(keys=[keys[p] for p in perm], values=torch.cat([seg[p] for p in perm]),
                           lengths=torch.cat([Lm[p] for p in perm])))
    same(KeyedJaggedTensor(keys=["other"] + keys, lengths=torch.cat([extra, lengths]),
                           values=torch.cat([torch.zeros(int(extra.sum()), dtype=torch.int64, device=DEV), values])))
    # int32 throughout takes the short route as well
    want32 = want
    got32 = m(KeyedJaggedTensor(keys=keys, values=values.to(torch.int32), lengths=lengths.to(torch.int32))).values()
    assert torch.equal(got32.view(torch.int16), want32.view(torch.int16))
    # with the flag, the first key order seen is kept (the reference's contract): general route
    m2 = QuantEBC(tables, False, DEV, output_dtype=torch.half, cache_features_order=True)
    m2._emb_modules[0].weights_dev.copy_(tbe.weights_dev)
    same(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths), m2)
    same(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths), m2)
    # a CPU KJT is refused by either route
    with pytest.raises(Exception):
        m(KeyedJaggedTensor(keys=keys, values=values.cpu(), lengths=lengths.cpu()))


@pytest.mark.parametrize("from_lengths", [True, False])
def test_forwards_in_flight_on_several_streams(from_lengths):
    """Independent requests on separate HIP streams (a serving loop): lookups of
    one module overlap on the GPU and every one gives the bits it gives alone.
    Large enough for the per-CU window kernel, whose blocks of consecutive
    launches then share the chip."""
    dev = DEV
    gen = torch.Generator(device="cpu").manual_seed(11)
    T, B, rows = 8, 2048, 20_000
    tables = [EmbeddingBagConfig(name=f"t{t}", embedding_dim=64, num_embeddings=rows, feature_names=[f"f{t}"],
                                 data_type=DataType.INT4, pooling=PoolingType.SUM) for t in range(T)]
    m = QuantEBC(tables, True, dev, output_dtype=torch.half)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, generator=gen).to(dev))
        for t in range(len(tbe.rows)):  # finite fp16 scale/bias headers
            tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=dev)
    keys = [f"f{t}" for t in range(T)]
    kjts = []
    for _ in range(4):
        lengths = torch.randint(0, 41, (T * B,), dtype=torch.int32, generator=gen)
        n = int(lengths.sum())
        values = torch.randint(0, rows, (n,), dtype=torch.int32, generator=gen).to(dev)
        weights = torch.rand(n, generator=gen).to(dev)
        if from_lengths:
            kjts.append(KeyedJaggedTensor(keys=keys, values=values, weights=weights, lengths=lengths.to(dev)))
        else:
            offsets = torch.zeros(T * B + 1, dtype=torch.int32)
            offsets[1:] = torch.cumsum(lengths, 0)
            kjts.append(KeyedJaggedTensor(keys=keys, values=values, weights=weights, offsets=offsets.to(dev)))
    alone = [m(k).values().clone() for k in kjts]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    got = []
    for k in range(48):
        with torch.cuda.stream(streams[k % 3]):
            got.append(m(kjts[k % 4]).values())
    torch.cuda.synchronize()
    for k, g in enumerate(got):
        assert torch.equal(g.view(torch.int16), alone[k % 4].view(torch.int16)), k
    assert all(t.out_of_range_count() == 0 for t in m._emb_modules)


def test_forwards_from_several_host_threads():
    """Three host threads, each with its own stream, call one module at once
    (ctypes releases the interpreter lock inside the C entry point)."""
    import threading

    gen = torch.Generator(device="cpu").manual_seed(12)
    T, B, rows = 6, 512, 5_000
    tables = [EmbeddingBagConfig(name=f"t{t}", embedding_dim=32, num_embeddings=rows, feature_names=[f"f{t}"],
                                 data_type=DataType.INT8, pooling=PoolingType.MEAN) for t in range(T)]
    m = QuantEBC(tables, False, DEV, output_dtype=torch.float)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, generator=gen).to(DEV))
        for t in range(len(tbe.rows)):
            tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    keys = [f"f{t}" for t in range(T)]
    kjts = []
    for _ in range(3):
        lengths = torch.randint(0, 30, (T * B,), dtype=torch.int32, generator=gen)
        values = torch.randint(0, rows, (int(lengths.sum()),), dtype=torch.int64, generator=gen).to(DEV)
        kjts.append(KeyedJaggedTensor(keys=keys, values=values, lengths=lengths.to(DEV)))
    alone = [m(k).values().clone() for k in kjts]
    torch.cuda.synchronize()
    results, errors = [None] * 3, []

    def worker(i):
        try:
            torch.cuda.set_device(DEV)
            s = torch.cuda.Stream()
            outs = []
            with torch.cuda.stream(s):
                for k in range(16):
                    outs.append(m(kjts[(i + k) % 3]).values())
            s.synchronize()
            results[i] = outs
        except Exception as e:  # surfaced in the main thread
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i in range(3):
        for k, o in enumerate(results[i]):
            assert torch.equal(o, alone[(i + k) % 3]), (i, k)


@pytest.mark.parametrize("seed", range(24))
def test_random_collections(seed):
    """Seeded random QuantEmbeddingBagCollections: tables of random type, width
    and pooling (one lookup operator per pooling), one to three features per
    table drawn from a small pool (so features are shared between tables and
    take the feature@table names), a KJT whose keys are a shuffled superset.
    Output keys follow the reference's naming rule; values match the oracle on
    the module's own packed bytes, bit for bit."""
    rng = np.random.default_rng(4000 + seed)
    pool = [f"f{i}" for i in range(6)]
    T = int(rng.integers(1, 9))
    weighted = bool(rng.integers(0, 2))
    out_dtype = [torch.float, torch.half][int(rng.integers(0, 2))]
    tables = []
    for t in range(T):
        names = [str(x) for x in rng.choice(pool, int(rng.integers(1, 4)), replace=False)]
        tables.append(EmbeddingBagConfig(
            name=f"t{t}", embedding_dim=int(rng.choice([16, 32, 64, 128, 192])),
            num_embeddings=int(rng.choice([3, 40, 700])), feature_names=names,
            data_type=[DataType.INT8, DataType.INT4, DataType.INT2, DataType.FP16][int(rng.integers(0, 4))],
            pooling=[PoolingType.SUM, PoolingType.MEAN][int(rng.integers(0, 2))]))
    m = QuantEBC(tables, weighted, DEV, output_dtype=out_dtype)
    gen = torch.Generator(device="cpu").manual_seed(seed)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, generator=gen).to(DEV))
        for t, ty in enumerate(tbe.weight_tys):
            if str(ty) in ("int8", "int4", "int2"):  # finite fp16 scale / bias
                tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
            else:                                    # finite fp16 payload: clear the top exponent bit
                tbe._rows_view(t)[:, 1::2] &= 0xBF
    used = sorted({f for t in tables for f in t.feature_names})
    keys = used + ["unused_a", "unused_b"][: int(rng.integers(0, 3))]
    rng.shuffle(keys)
    rows_of = {k: min([t.num_embeddings for t in tables if k in t.feature_names], default=5) for k in keys}
    B = int(rng.choice([1, 5, 64, 300]))
    kjt = random_kjt(rng, keys, [rows_of[k] for k in keys], B=B, max_len=int(rng.choice([2, 9, 30])),
                     weighted=weighted, idt=[torch.int32, torch.int64][int(rng.integers(0, 2))])
    got = m(kjt)
    # naming rule (torchrec/modules/embedding_modules.py:75-94): a feature of
    # several tables is named feature@table; order = tables grouped by pooling
    count = {f: sum(f in t.feature_names for t in tables) for f in used}
    grouped = [t for p in (PoolingType.SUM, PoolingType.MEAN) for t in tables if t.pooling == p]
    if tables[0].pooling == PoolingType.MEAN:  # groups appear in order of first use
        grouped = [t for p in (PoolingType.MEAN, PoolingType.SUM) for t in tables if t.pooling == p]
    want_keys = [f if count[f] == 1 else f"{f}@{t.name}" for t in grouped for f in t.feature_names]
    assert got.keys() == want_keys
    assert got.length_per_key() == [t.embedding_dim for t in grouped for _ in t.feature_names]
    order = [kjt.keys().index(k) for k in m._feature_names]
    perm = kjt.permute(order)
    ids, offs = perm.values().cpu().numpy(), perm.offsets().cpu().numpy().astype(np.int64)
    psw = perm.weights().cpu().numpy() if weighted else None
    col, f0 = 0, 0
    gv = got.values().cpu().numpy()
    assert gv.shape == (B, sum(got.length_per_key()))
    for tbe, nf in zip(m._emb_modules, m._feature_splits):
        o = offs[f0 * B:(f0 + nf) * B + 1]
        sl = slice(int(o[0]), int(o[-1]))
        want = O.tbe_forward(oracle_store_of(tbe), tbe.feature_table_map, B, ids[sl].astype(np.int64), o - o[0],
                             None if psw is None else psw[sl], int(tbe.pooling_mode),
                             O.FP16 if out_dtype == torch.half else O.FP32)
        assert bits_equal(np.ascontiguousarray(gv[:, col:col + tbe.total_D]), want) == 0, (seed, col)
        col += tbe.total_D
        f0 += nf


@pytest.mark.parametrize("seed", range(16))
def test_random_sequence_collections(seed):
    """Seeded random QuantEmbeddingCollections (one lookup operator per weight
    type, shared features, shuffled superset of keys, need_indices): every
    output JaggedTensor carries its key's lengths and, row by row, the
    dequantized rows of the oracle on the module's own packed bytes."""
    rng = np.random.default_rng(6000 + seed)
    pool = [f"f{i}" for i in range(5)]
    T = int(rng.integers(1, 7))
    dim = int(rng.choice([16, 32, 64, 128]))
    need_indices = bool(rng.integers(0, 2))
    out_dtype = [torch.float, torch.half][int(rng.integers(0, 2))]
    tables = []
    for t in range(T):
        names = [str(x) for x in rng.choice(pool, int(rng.integers(1, 3)), replace=False)]
        tables.append(EmbeddingConfig(
            name=f"t{t}", embedding_dim=dim, num_embeddings=int(rng.choice([3, 40, 700])), feature_names=names,
            data_type=[DataType.INT8, DataType.INT4, DataType.INT2, DataType.FP16][int(rng.integers(0, 4))]))
    m = QuantEC(tables, DEV, need_indices=need_indices, output_dtype=out_dtype)
    gen = torch.Generator(device="cpu").manual_seed(seed)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, generator=gen).to(DEV))
        for t, ty in enumerate(tbe.weight_tys):
            if str(ty) in ("int8", "int4", "int2"):
                tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
            else:
                tbe._rows_view(t)[:, 1::2] &= 0xBF
    used = sorted({f for t in tables for f in t.feature_names})
    keys = used + ["unused_a", "unused_b"][: int(rng.integers(0, 3))]
    rng.shuffle(keys)
    rows_of = {k: min([t.num_embeddings for t in tables if k in t.feature_names], default=5) for k in keys}
    B = int(rng.choice([1, 5, 64, 300]))
    kjt = random_kjt(rng, keys, [rows_of[k] for k in keys], B=B, max_len=int(rng.choice([2, 9, 30])),
                     idt=[torch.int32, torch.int64][int(rng.integers(0, 2))])
    got = m(kjt)
    # Output names are made per lookup operator (torchrec/quant/embedding_modules.py:872-877):
    # a feature is named feature@table only where it is shared INSIDE its
    # weight-type group; the same plain name from two groups lands on one
    # dict entry and the later group's tensor stays.
    jd = kjt.to_dict()
    expected = {}
    f = 0
    for tbe, nf in zip(m._emb_modules, m._feature_splits):
        group_features = m._feature_names[f:f + nf]
        for k in range(nf):
            feature = group_features[k]
            t = tbe.feature_table_map[k]
            name = feature if group_features.count(feature) == 1 else f"{feature}@{tbe.embedding_names[t]}"
            expected[name] = (tbe, t, feature)
        f += nf
    assert set(got.keys()) == set(expected)
    for name, (tbe, t, feature) in expected.items():
        jt = got[name]
        ids = jd[feature].values().cpu().numpy()
        want = O.tbe_forward(oracle_store_of(tbe), [t], 1, ids, np.array([0, len(ids)], dtype=ids.dtype), None,
                             O.NONE, O.FP16 if out_dtype == torch.half else O.FP32)
        assert jt.values().dtype == out_dtype
        assert bits_equal(jt.values().cpu().numpy(), want) == 0, (seed, name)
        assert torch.equal(jt.lengths(), jd[feature].lengths())
        if need_indices:
            assert torch.equal(jt.weights(), jd[feature].values())
        else:
            assert jt.weights_or_none() is None
    # the accessor names tables over the whole collection (:879-881)
    count = {f_: sum(f_ in t.feature_names for t in tables) for f_ in used}
    assert m.embedding_names_by_table() == [
        [f_ if count[f_] == 1 else f"{f_}@{t.name}" for f_ in t.feature_names] for t in tables]


def test_deepcopy_of_a_used_collection():
    """A collection that has already looked up (and so holds launch plans) can
    be deep-copied; the copy has its own bytes and gives the same outputs."""
    import copy

    rng = np.random.default_rng(21)
    tables = [EmbeddingBagConfig(name=f"t{i}", embedding_dim=32, num_embeddings=60, feature_names=[f"f{i}"],
                                 data_type=DataType.INT4) for i in range(3)]
    m = QuantEBC(tables, False, DEV, output_dtype=torch.float)
    for tbe in m._emb_modules:
        tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8).to(DEV))
        for t in range(len(tbe.rows)):
            tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    kjt = random_kjt(rng, ["f0", "f1", "f2"], [60] * 3, B=17, max_len=6)
    before = m(kjt).values().clone()
    twin = copy.deepcopy(m)
    assert torch.equal(twin(kjt).values(), before)
    twin._emb_modules[0].weights_dev.zero_()
    assert torch.equal(m(kjt).values(), before)           # the original kept its bytes
    assert not torch.equal(twin(kjt).values(), before)
    # the copy's state_dict tensors view the copy's buffer, as the original's view the original's
    sd = twin.state_dict()
    assert all(not v.view(torch.uint8).any() for k, v in sd.items() if k.endswith(".weight"))


def test_qebc_shared_feature_and_registered_operators_take_the_general_route():
    """A feature that feeds two tables makes the module's feature names repeat ([a, a, b]): a KJT
    whose keys happen to equal that list must not take the short route (it would read the second
    table's bags from the second key).  Registered operators are called as modules and give the
    same bits as unregistered ones."""
    torch.manual_seed(5)
    B = 40
    tables = [EmbeddingBagConfig(name="t0", embedding_dim=32, num_embeddings=100, feature_names=["a"], data_type=DataType.INT4),
              EmbeddingBagConfig(name="t1", embedding_dim=64, num_embeddings=200, feature_names=["a", "b"], data_type=DataType.INT8)]
    m = QuantEBC(tables, False, DEV, output_dtype=torch.half)
    assert m._feature_names == ["a", "a", "b"] and len(m._emb_modules) == 1
    tbe = m._emb_modules[0]
    tbe.weights_dev.copy_(torch.randint(0, 256, tbe.weights_dev.shape, dtype=torch.uint8, device=DEV))
    for t in range(2):
        tbe._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    la = torch.randint(0, 6, (B,), dtype=torch.int64, device=DEV)
    lb = torch.randint(0, 6, (B,), dtype=torch.int64, device=DEV)
    va = torch.randint(0, 100, (int(la.sum()),), dtype=torch.int64, device=DEV)
    vb = torch.randint(0, 200, (int(lb.sum()),), dtype=torch.int64, device=DEV)
    kjt = KeyedJaggedTensor(keys=["a", "b"], values=torch.cat([va, vb]), lengths=torch.cat([la, lb]))
    want = m(kjt).values()
    # the same bags written out once per use of the feature: keys == the module's feature names
    dup = KeyedJaggedTensor(keys=["a", "a", "b"], values=torch.cat([va, va, vb]), lengths=torch.cat([la, la, lb]))
    got = m(dup).values()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # oracle on the module's packed bytes
    off = np.zeros(3 * B + 1, dtype=np.int64)
    off[1:] = np.cumsum(torch.cat([la, la, lb]).cpu().numpy())
    ref = O.tbe_forward(oracle_store_of(tbe), [0, 1, 1], B, torch.cat([va, va, vb]).cpu().numpy(), off, None, O.SUM, O.FP16)
    assert bits_equal(want.cpu().numpy(), ref) == 0
    # a stride that disagrees with the lengths is not silently accepted by the short route
    single = QuantEBC(tables[1:], False, DEV, output_dtype=torch.half)
    single._emb_modules[0].weights_dev.copy_(torch.randint(0, 256, single._emb_modules[0].weights_dev.shape, dtype=torch.uint8, device=DEV))
    single._emb_modules[0]._rows_view(0)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    ok = KeyedJaggedTensor(keys=["a", "b"], values=torch.cat([va, vb]) % 200, lengths=torch.cat([la, lb]))
    base = single(ok).values()
    with_stride = KeyedJaggedTensor(keys=["a", "b"], values=torch.cat([va, vb]) % 200, lengths=torch.cat([la, lb]), stride=B)
    assert torch.equal(single(with_stride).values().view(torch.int16), base.view(torch.int16))
    # registered operators: hooks fire, same bits
    reg = QuantEBC(tables, False, DEV, output_dtype=torch.half, register_tbes=True)
    reg._emb_modules[0].weights_dev.copy_(tbe.weights_dev)
    fired = []
    reg.tbes[0].register_forward_hook(lambda mod, args, out: fired.append(out.shape))
    got = reg(kjt).values()
    assert fired == [(B, 32 + 64 + 64)] and torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_qec_prepared_flags_and_registered_operators_give_the_same_rows():
    """``__use_unflattened_lengths_for_batching``, ``__use_batching_hinted_output`` off,
    ``__remove_stbe_padding`` and ``register_tbes`` change how the lookup is wrapped, not its rows."""
    from torchrec_amd.quant import embedding_modules as qm

    rng = np.random.default_rng(21)
    t = [EmbeddingConfig(name="t1", embedding_dim=32, num_embeddings=50, feature_names=["f1", "f2"], data_type=DataType.INT8),
         EmbeddingConfig(name="t2", embedding_dim=32, num_embeddings=70, feature_names=["f3"], data_type=DataType.INT4)]
    base = QuantEC(t, DEV, output_dtype=torch.half, need_indices=True)
    for op in base._emb_modules:
        op.weights_dev.copy_(torch.randint(0, 256, op.weights_dev.shape, dtype=torch.uint8, device=DEV))
        for i in range(len(op.rows)):
            op._rows_view(i)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    kjt = random_kjt(rng, ["f3", "f1", "f2"], [70, 50, 50], B=17, max_len=6)
    want = base(kjt)
    variants = []
    for attr, value in ((qm.MODULE_ATTR_USE_UNFLATTENED_LENGTHS_FOR_BATCHING, True),
                        (qm.MODULE_ATTR_USE_BATCHING_HINTED_OUTPUT, False),
                        (qm.MODULE_ATTR_REMOVE_STBE_PADDING_BOOL, True)):
        m = QuantEC(t, DEV, output_dtype=torch.half, need_indices=True)
        setattr(m, attr, value)
        variants.append(m)
    variants.append(QuantEC(t, DEV, output_dtype=torch.half, need_indices=True, register_tbes=True))
    fired = []
    for op in variants[-1].tbes:
        op.register_forward_pre_hook(lambda mod, args: fired.append(1))
    for m in variants:
        for src, dst in zip(base._emb_modules, m._emb_modules):
            dst.weights_dev.copy_(src.weights_dev)
        got = m(random_kjt(np.random.default_rng(21), ["f3", "f1", "f2"], [70, 50, 50], B=17, max_len=6))
        assert got.keys() == want.keys() if hasattr(got, "keys") else True
        for k in ("f1", "f2", "f3"):
            assert torch.equal(got[k].values().view(torch.int16), want[k].values().view(torch.int16))
            assert torch.equal(got[k].lengths(), want[k].lengths()) and torch.equal(got[k].weights(), want[k].weights())
    assert len(fired) == 2


@pytest.mark.parametrize("observer", ["none", "hook", "pre_hook", "global", "replaced", "traced"])
def test_registered_operator_is_called_where_the_call_can_be_seen(observer):
    """A registered operator is launched directly only while nothing could see the module call; an observer added
    after calls that were launched directly sees every later one."""
    tables = [EmbeddingBagConfig(name="t", embedding_dim=32, num_embeddings=50, feature_names=["a"], data_type=DataType.INT8)]
    reg = QuantEBC(tables, False, DEV, output_dtype=torch.half, register_tbes=True)
    op = reg.tbes[0]
    op.weights_dev.zero_()
    op._rows_view(0)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
    kjt = KeyedJaggedTensor(keys=["a"], values=torch.arange(7, device=DEV), lengths=torch.tensor([3, 0, 4], device=DEV))
    want = reg(kjt).values().clone()
    seen, handle = [], None
    forward = type(op).forward
    if observer == "hook":
        handle = op.register_forward_hook(lambda mod, args, out: seen.append(mod))
    elif observer == "pre_hook":
        handle = op.register_forward_pre_hook(lambda mod, args: seen.append(mod))
    elif observer == "global":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, args, out: seen.append(mod))
    elif observer == "replaced":
        op.forward = lambda *args, **kwargs: (seen.append(op), forward(op, *args, **kwargs))[1]
    plain = torch.nn.Module.__call__
    try:
        if observer == "traced":
            torch.nn.Module.__call__ = lambda mod, *args, **kwargs: (seen.append(mod), plain(mod, *args, **kwargs))[1]
        got = reg(kjt).values()
    finally:
        torch.nn.Module.__call__ = plain
        if handle is not None:
            handle.remove()
    assert (op in seen) == (observer != "none")
    assert torch.equal(got, want)


@pytest.mark.parametrize("first", ["ab", "ba"])
def test_kept_features_order_with_and_without_the_short_route(first):
    """``cache_features_order``: the first key order seen holds for every later call, whichever way the operator is
    launched (a hook keeps the call off the short route)."""
    tables = [EmbeddingBagConfig(name=f"t{k}", embedding_dim=32, num_embeddings=50, feature_names=[k], data_type=DataType.INT8)
              for k in "ab"]
    got = {}
    for hooked in (False, True):
        q = QuantEBC(tables, False, DEV, output_dtype=torch.half, register_tbes=True, cache_features_order=True)
        op = q.tbes[0]
        g = torch.Generator(device="cuda").manual_seed(5)
        op.weights_dev.random_(0, 256, generator=g)
        for t in range(2):
            op._rows_view(t)[:, 0:4] = torch.tensor([0x00, 0x2C, 0x00, 0xAC], dtype=torch.uint8, device=DEV)
        if hooked:
            op.register_forward_hook(lambda mod, args, out: None)
        lengths = torch.tensor([3, 0, 4, 1, 2, 2], device=DEV)
        ids = torch.arange(12, device=DEV) * 4
        got[hooked] = [q(KeyedJaggedTensor(keys=list(keys), values=ids, lengths=lengths)).values().clone()
                       for keys in (first, "ab", "ba", "ab")]
    assert all(torch.equal(x, y) for x, y in zip(got[False], got[True]))
    assert all(torch.equal(x, got[False][0]) for x in got[False])


@pytest.mark.parametrize("weight_dtype", [torch.qint8, torch.quint4x2, torch.quint2x4, torch.half, torch.float])
@pytest.mark.parametrize("empty", [0, 1, 2])
def test_from_float_with_a_table_of_no_rows(weight_dtype, empty):
    """A table without rows among others, in every place: converted like the rest (its lookup is refused, as ever)."""
    rows = [7, 5, 9]
    rows[empty] = 0
    tables = [EmbeddingBagConfig(name=f"t{t}", embedding_dim=32, num_embeddings=n, feature_names=[f"f{t}"],
                                 weight_init_min=-1.0, weight_init_max=1.0) for t, n in enumerate(rows)]
    ebc = EmbeddingBagCollection(tables=tables, device=DEV)
    for dtype in (torch.float, torch.half):
        ebc = ebc.to(dtype)
        ebc.qconfig = qconfig(weight_dtype, torch.float)
        qebc = QuantEBC.from_float(ebc)
        want = {}
        quantize_state_dict(ebc, want, {t.name: t.data_type for t in qebc.embedding_bag_configs()})
        (op,) = qebc._emb_modules
        for name, n, got in zip(op.embedding_names, op.rows, op.split_embedding_weights()):
            assert n == rows[int(name[1:])]
            for g, w in zip(got, want[name]):
                assert (g is None and w is None) or torch.equal(g, w)


@pytest.mark.parametrize("registered,observer", [(True, "pre_hook"), (True, "replaced"), (False, "replaced"), (True, "class"),
                                                 (True, "none")])
@pytest.mark.parametrize("counts", [False, True])
def test_sequence_lookups_that_can_be_seen_get_offsets(registered, observer, counts):
    """Whatever looks at, or stands in for, the operators of a sequence collection is called with the ids and the
    bags' offsets, whether the KJT carries its per-key counts or not."""
    table = EmbeddingConfig(name="t", embedding_dim=16, num_embeddings=30, feature_names=["f", "g"], data_type=DataType.INT8)
    qec = QuantEC([table], DEV, output_dtype=torch.half, register_tbes=registered)
    (op,) = qec._emb_modules
    seen = []
    own = type(op).forward

    def stand_in(indices, offsets, feature_positions=None, batch_size=None, out=None):
        seen.append(offsets)
        return own(op, indices, offsets, feature_positions=feature_positions, batch_size=batch_size, out=out)

    kjt = random_kjt(np.random.default_rng(5), ["g", "f"], [30, 30], B=9, max_len=4)
    if counts:
        kjt.length_per_key()
    want = qec(kjt)
    if observer == "pre_hook":
        op.register_forward_pre_hook(lambda m, args, kw: seen.append(kw["offsets"]), with_kwargs=True)
    elif observer == "replaced":
        op.forward = stand_in
    elif observer == "class":
        op.__class__ = type("Other", (type(op),), {"forward": lambda self, **kw: stand_in(**kw)})
    kjt = random_kjt(np.random.default_rng(5), ["g", "f"], [30, 30], B=9, max_len=4)
    if counts:
        kjt.length_per_key()
    got = qec(kjt)
    assert all(torch.equal(got[k].values(), want[k].values()) for k in "fg")
    assert len(seen) == (observer != "none") and all(torch.equal(x, kjt.offsets()) for x in seen)
