"""Managed-collision remap and the quantized collection behind it.  Expected
ids are computed with numpy's searchsorted, i.e. the reference's formula
(torchrec/modules/mc_modules.py:959-989) restated on the host."""
import numpy as np
import pytest
import torch
import torch.quantization as quant

from torchrec_amd import KeyedJaggedTensor, ops
from torchrec_amd.modules.embedding_configs import EmbeddingConfig, QuantConfig
from torchrec_amd.modules.embedding_modules import EmbeddingCollection
from torchrec_amd.modules.mc_embedding_modules import ManagedCollisionEmbeddingCollection
from torchrec_amd.modules.mc_modules import ManagedCollisionCollection, MCHManagedCollisionModule
from torchrec_amd.quant import QuantManagedCollisionEmbeddingCollection as QuantMCEC

IMAX = np.iinfo(np.int64).max


def ref_remap(values, sorted_ids, mapping, miss):
    idx = np.searchsorted(sorted_ids[:-1], values)
    hit = sorted_ids[idx] == values
    return np.where(hit, mapping[idx], miss)


def make_table(rng, size, filled):
    raw = np.sort(rng.choice(10**9, filled, replace=False)).astype(np.int64)
    sorted_ids = np.full(size, IMAX, dtype=np.int64)
    sorted_ids[:filled] = raw
    mapping = rng.permutation(size).astype(np.int64)
    return sorted_ids, mapping


@pytest.mark.parametrize("size,filled", [(1, 0), (2, 1), (64, 63), (1000, 400)])
def test_mch_remap_host(size, filled):
    rng = np.random.default_rng(size)
    sorted_ids, mapping = make_table(rng, size, filled)
    values = np.concatenate([rng.choice(sorted_ids[:max(filled, 1)], 50), rng.integers(0, 10**9, 50), [IMAX, 0]]).astype(np.int64)
    got = ops.mch_remap(torch.from_numpy(values), torch.from_numpy(sorted_ids), torch.from_numpy(mapping), size - 1)
    assert np.array_equal(got.numpy(), ref_remap(values, sorted_ids, mapping, size - 1))


@pytest.mark.gpu
@pytest.mark.parametrize("idt", [np.int32, np.int64])
@pytest.mark.parametrize("size,filled", [(1, 0), (2, 1), (64, 63), (100_000, 60_000)])
def test_mch_remap_kernel(idt, size, filled):
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(size + 1)
    sorted_ids, mapping = make_table(rng, size, filled)
    hits = rng.choice(sorted_ids[:max(filled, 1)], 5000)
    values = np.concatenate([hits, rng.integers(0, 10**9, 5000), [0, 10**9]])
    if idt == np.int64:
        values = np.concatenate([values, [IMAX, -5]])
    values = values.astype(idt)
    got = ops.mch_remap(torch.from_numpy(values).to(dev), torch.from_numpy(sorted_ids).to(dev),
                        torch.from_numpy(mapping).to(dev), size - 1)
    assert got.dtype == torch.from_numpy(values).dtype
    assert np.array_equal(got.cpu().numpy(), ref_remap(values.astype(np.int64), sorted_ids, mapping, size - 1).astype(idt))
    assert np.array_equal(got.cpu().numpy(), ops.mch_remap(torch.from_numpy(values), torch.from_numpy(sorted_ids),
                                                           torch.from_numpy(mapping), size - 1).numpy())


def build_mcec(dev):
    configs = [
        EmbeddingConfig(name="t1", embedding_dim=16, num_embeddings=40, feature_names=["f1", "f2"]),
        EmbeddingConfig(name="t2", embedding_dim=16, num_embeddings=30, feature_names=["f3"]),
    ]
    mods = {c.name: MCHManagedCollisionModule(c.num_embeddings, dev) for c in configs}
    mods["t1"].set_id_table(torch.tensor([1000, 5, 77777, 123456789]))
    mods["t2"].set_id_table(torch.tensor([9, 8, 7]), rows=torch.tensor([20, 21, 22]))
    mcc = ManagedCollisionCollection(mods, configs)
    return ManagedCollisionEmbeddingCollection(EmbeddingCollection(configs, dev), mcc, return_remapped_features=True)


def test_collection_remap_and_errors_host():
    cpu = torch.device("cpu")
    m = build_mcec(cpu).eval()
    # keys in a different order than the tables' features
    kjt = KeyedJaggedTensor(keys=["f3", "f1", "f2"], values=torch.tensor([9, 1, 7, 5, 1000, 2, 123456789, 77777]),
                            lengths=torch.tensor([2, 1, 1, 1, 2, 1]))
    out = m._managed_collision_collection(kjt)
    assert out.keys() == ["f1", "f2", "f3"]
    assert out.lengths().tolist() == [1, 1, 2, 1, 2, 1]
    # t1 sorted raw ids: 5, 1000, 77777, 123456789 -> rows 1, 0, 2, 3; miss -> 39.  t2: 7->22, 8->21, 9->20; miss -> 29
    assert out.values().tolist() == [1, 0, 39, 3, 2, 20, 29, 22]
    emb, remapped = m(kjt)
    assert set(emb.keys()) == {"f1", "f2", "f3"} and remapped.values().tolist() == out.values().tolist()
    with pytest.raises(ValueError):
        ManagedCollisionCollection({}, m._managed_collision_collection.embedding_configs())
    with pytest.raises(AssertionError):
        ManagedCollisionCollection({"t1": MCHManagedCollisionModule(7, cpu), "t2": MCHManagedCollisionModule(30, cpu)},
                                   m._managed_collision_collection.embedding_configs())
    m.train()
    with pytest.raises(NotImplementedError):
        m._managed_collision_collection(kjt)
    # the id table travels through a state_dict
    sd = m._managed_collision_collection.state_dict()
    assert "_managed_collision_modules.t1._mch_sorted_raw_ids" in sd and "_managed_collision_modules.t2._mch_remapped_ids_mapping" in sd


@pytest.mark.gpu
def test_quant_mcec_matches_float():
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    m = build_mcec(dev).eval()
    kjt = KeyedJaggedTensor(keys=["f3", "f1", "f2"],
                            values=torch.tensor([9, 1, 7, 5, 1000, 2, 123456789, 77777], device=dev),
                            lengths=torch.tensor([2, 1, 1, 1, 2, 1], device=dev))
    with torch.no_grad():
        want, want_kjt = m(kjt)
    m.qconfig = QuantConfig(activation=quant.PlaceholderObserver.with_args(dtype=torch.float),
                            weight=quant.PlaceholderObserver.with_args(dtype=torch.qint8))
    q = QuantMCEC.from_float(m)
    got, got_kjt = q(kjt)
    assert torch.equal(got_kjt.values(), want_kjt.values()) and got_kjt.keys() == want_kjt.keys()
    assert got_kjt.values().tolist() == [1, 0, 39, 3, 2, 20, 29, 22]
    for k in ("f1", "f2", "f3"):
        assert torch.equal(got[k].lengths(), want[k].lengths())
        assert torch.allclose(got[k].values(), want[k].values(), atol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
def test_collection_remaps_all_keys_in_one_launch(idt):
    """The collection's GPU path (every key in one launch) against numpy's
    searchsorted per table: two features on one table, one key without ids, a
    key order that differs from the tables'."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(11)
    sizes = {"t1": (500, 300), "t2": (64, 63), "t3": (2000, 1500)}
    configs = [EmbeddingConfig(name="t1", embedding_dim=8, num_embeddings=500, feature_names=["a", "b"]),
               EmbeddingConfig(name="t2", embedding_dim=8, num_embeddings=64, feature_names=["c"]),
               EmbeddingConfig(name="t3", embedding_dim=8, num_embeddings=2000, feature_names=["d"])]
    modules, tables = {}, {}
    for name, (size, filled) in sizes.items():
        raw = rng.choice(2**31 - 2, filled, replace=False).astype(np.int64)
        rows = rng.permutation(size - 1)[:filled].astype(np.int64)
        mod = MCHManagedCollisionModule(size, dev)
        mod.set_id_table(torch.from_numpy(raw), torch.from_numpy(rows))
        modules[name] = mod
        tables[name] = (raw, rows, size - 1)
    mcc = ManagedCollisionCollection(modules, configs).eval()
    keys, B = ["d", "a", "c", "b"], 19
    lengths = rng.integers(0, 9, len(keys) * B)
    lengths[2 * B:3 * B] = 0  # "c" has no ids at all
    table_of = {"a": "t1", "b": "t1", "c": "t2", "d": "t3"}
    vals = []
    for k, key in enumerate(keys):
        raw = tables[table_of[key]][0]
        n = int(lengths[k * B:(k + 1) * B].sum())
        known = rng.choice(raw, n)
        unknown = rng.integers(0, 2**31 - 2, n)
        vals.append(np.where(rng.random(n) < 0.6, known, unknown))
    values = np.concatenate(vals).astype(np.int64)
    kjt = KeyedJaggedTensor(keys=keys, values=torch.from_numpy(values).to(idt).to(dev),
                            lengths=torch.from_numpy(lengths).to(dev))
    out = mcc(kjt)
    assert out.keys() == ["a", "b", "c", "d"] and out.values().dtype == idt
    per_key = dict(zip(keys, vals))
    want = []
    for key in out.keys():
        raw, rows, miss = tables[table_of[key]]
        lut = dict(zip(raw.tolist(), rows.tolist()))
        want += [lut.get(int(v), miss) for v in per_key[key]]
    assert out.values().cpu().tolist() == want
    assert out.lengths().cpu().tolist() == np.concatenate(
        [lengths[keys.index(k) * B:(keys.index(k) + 1) * B] for k in out.keys()]).tolist()


def _remap_numpy(values, sorted_ids, mapping, miss):
    """First index in [0, size - 1] whose entry is >= the id, searched over the first size - 1 entries."""
    at = np.searchsorted(sorted_ids[:-1], values)
    return np.where(sorted_ids[at] == values, mapping[at], miss)


@pytest.mark.gpu
# Around the four entries of a read, the 512 pivots of a block, and segments of many entries.
@pytest.mark.parametrize("size", [1, 2, 3, 4, 5, 9, 511, 512, 513, 514, 1026, 5000, 70_001])
@pytest.mark.parametrize("kind", ["even", "clustered", "geometric", "half empty", "repeats", "delimiter first"])
def test_remap_search(size, kind):
    rng = np.random.default_rng(size)
    if kind == "clustered":
        ids = np.concatenate([c + rng.integers(0, 3 * size, size) for c in rng.integers(-2**62, 2**62, 7)])[:size]
    elif kind == "geometric":
        ids = np.exp(rng.uniform(0, 43, size)).astype(np.int64)
    elif kind == "repeats":
        ids = rng.integers(0, max(1, size // 3), size)
    else:
        ids = rng.integers(-2**40, 2**40, size)
    table = np.sort(ids.astype(np.int64))
    if kind == "half empty":
        table[size // 2:] = np.iinfo(np.int64).max
    table[-1] = np.iinfo(np.int64).max
    if kind == "delimiter first":  # (the last entry is compared, never searched: it may be the smallest)
        table[-1] = -2**50
    mapping = rng.permutation(size).astype(np.int64)
    values = np.concatenate([table, table - 1, table + np.where(table == np.iinfo(np.int64).max, 0, 1),
                             rng.integers(-2**41, 2**41, 1500), [np.iinfo(np.int64).min, np.iinfo(np.int64).max, 0]])
    dev = torch.device("cuda:0")
    got = ops.mch_remap(torch.from_numpy(values).to(dev), torch.from_numpy(table).to(dev), torch.from_numpy(mapping).to(dev), 77)
    assert np.array_equal(got.cpu().numpy(), _remap_numpy(values, table, mapping, 77))


@pytest.mark.gpu
@pytest.mark.parametrize("K,B", [(1, 1), (3, 5), (70, 9), (256, 2), (257, 2)])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("given", ["lengths", "offsets"])
def test_collection_remap_many_keys(K, B, shuffled, given):
    """More keys than a launch has tables, more than the one-launch route takes; keys without ids."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(K)
    configs = [EmbeddingConfig(name=f"t{k}", embedding_dim=4, num_embeddings=50 + k, feature_names=[f"f{k}"]) for k in range(K)]
    modules, tables = {}, {}
    for c in configs:
        raw = rng.choice(10_000, 30, replace=False)
        modules[c.name] = MCHManagedCollisionModule(c.num_embeddings, dev)
        modules[c.name].set_id_table(torch.from_numpy(raw), torch.arange(30) * 1)
        tables[c.feature_names[0]] = (modules[c.name]._mch_sorted_raw_ids.cpu().numpy(),
                                      modules[c.name]._mch_remapped_ids_mapping.cpu().numpy(), c.num_embeddings - 1)
    mcc = ManagedCollisionCollection(modules, configs).eval()
    keys = [f"f{k}" for k in (rng.permutation(K) if shuffled else range(K))]
    lengths = rng.integers(0, 12, (K, B))
    lengths[rng.random(K) < 0.3] = 0
    values = [rng.integers(0, 10_000, n) for n in lengths.sum(1)]
    weights = torch.rand(int(lengths.sum()), device=dev)
    bags = torch.from_numpy(lengths.reshape(-1)).to(dev)
    if given == "offsets":
        bags = ops.asynchronous_complete_cumsum(bags)
    kjt = KeyedJaggedTensor(keys=keys, values=torch.from_numpy(np.concatenate(values)).to(dev), weights=weights, **{given: bags})
    out = mcc(kjt)
    order = [keys.index(f"f{k}") for k in range(K)]
    assert out.keys() == [f"f{k}" for k in range(K)]
    want = np.concatenate([_remap_numpy(values[i], *tables[keys[i]]) for i in order])
    assert np.array_equal(out.values().cpu().numpy(), want)
    assert np.array_equal(out.lengths().cpu().numpy(), lengths[order].reshape(-1))
    starts = np.concatenate([[0], np.cumsum(lengths.sum(1))])
    assert torch.equal(out.weights(), torch.cat([weights[starts[i]:starts[i + 1]] for i in order]))
    assert out.length_per_key() == lengths.sum(1)[order].tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("keys", [["a", "b"], ["b", "a"]])
@pytest.mark.parametrize("given", ["lengths", "offsets"])
def test_collection_remap_refuses_what_its_kernels_cannot_read(keys, given):
    """Values that are no int32 / int64 ids, and tables of another type or size, on every route of the collection."""
    dev = torch.device("cuda:0")
    configs = [EmbeddingConfig(name=f"t{f}", embedding_dim=4, num_embeddings=20, feature_names=[f]) for f in "ab"]
    bags = torch.tensor([1, 2, 0, 1] if given == "lengths" else [0, 1, 3, 3, 4], device=dev)

    def collection():
        modules = {c.name: MCHManagedCollisionModule(20, dev) for c in configs}
        return ManagedCollisionCollection(modules, configs).eval()

    for dtype in (torch.float32, torch.float64):
        with pytest.raises(TypeError, match="int32 or int64"):
            collection()(KeyedJaggedTensor(keys=keys, values=torch.ones(4, dtype=dtype, device=dev), **{given: bags}))
    ids = torch.arange(4, device=dev)
    for name in ("_mch_sorted_raw_ids", "_mch_remapped_ids_mapping"):
        for bad in (lambda t: t.to(torch.int32), lambda t: t[:-1], lambda t: t.repeat_interleave(2)[::2]):
            mcc = collection()
            module = mcc._managed_collision_modules["tb"]
            setattr(module, name, bad(getattr(module, name)))
            with pytest.raises(AssertionError):
                mcc(KeyedJaggedTensor(keys=keys, values=ids, **{given: bags}))


def _hash(ids, size):
    return (ids * 7 + 3) % size


class _HashModule(torch.nn.Module):
    def forward(self, ids, size):
        return _hash(ids, size)


# CPU tensors stand for a GPU's: what is asked of the features here is only where their ids are.
class _OnDevice:
    def __init__(self, values):
        self._values = values

    def values(self):
        return self

    is_cuda = True

    def get_device(self):
        return self._values.get_device()

    def keys(self):
        return ["f"]


@pytest.mark.parametrize("hash_func", [None, _hash, _HashModule()], ids=["none", "function", "module"])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)])
def test_input_hash(hash_func, device):
    """An input hash may be any callable, a module too; ids are hashed before they are remapped."""
    rng = np.random.default_rng(3)
    sorted_ids, mapping = make_table(rng, 200, 150)
    size = 10**9
    dev = torch.device(device)
    mc = MCHManagedCollisionModule(200, dev, input_hash_size=size, input_hash_func=hash_func).eval()
    mc._mch_sorted_raw_ids.copy_(torch.from_numpy(sorted_ids))
    mc._mch_remapped_ids_mapping.copy_(torch.from_numpy(mapping))
    table = EmbeddingConfig(name="t", embedding_dim=8, num_embeddings=200, feature_names=["f"])
    collection = ManagedCollisionCollection({"t": mc}, [table]).eval()
    tables = collection._one_launch_tables(_OnDevice(mc._mch_sorted_raw_ids))
    assert (tables is None) == (hash_func is not None)
    # (7 * x + 3) % 10^9 = id: every other id is a known one
    inverse = pow(7, -1, size)
    known = rng.choice(sorted_ids[:150], 60)
    raw = known if hash_func is None else (known - 3) * inverse % size
    values = np.stack([raw, rng.integers(0, size, 60)], 1).reshape(-1)
    kjt = KeyedJaggedTensor(keys=["f"], values=torch.from_numpy(values).to(dev),
                            lengths=torch.full((40,), 3, dtype=torch.int64, device=dev))
    got = collection(kjt).values().cpu().numpy()
    want = ref_remap(values if hash_func is None else (values * 7 + 3) % size, sorted_ids, mapping, 199)
    assert np.array_equal(got, want)
    assert (want != 199).sum() >= 60
