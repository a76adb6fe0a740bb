"""KeyedTensor.regroup / regroup_as_dict: the cases of the reference's test
(torchrec/sparse/tests/test_keyed_tensor.py:82-128 single and multiple
KeyedTensors, :306-332 duplicate keys), on the host and, for the one-launch
column-copy kernel, on the GPU against plain slicing."""
import numpy as np
import pytest
import torch

from torchrec_amd import KeyedTensor
from torchrec_amd.sparse.jagged_tensor import _regroup_keyed_tensors, permute_multi_embedding, regroup_kts

DEVICES = ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("dev", DEVICES)
def test_regroup_single_kt(dev):
    tensors = [torch.randn(2, 3, device=dev) for _ in range(5)]
    kt = KeyedTensor.from_tensor_list([f"dense_{i}" for i in range(5)], tensors, 1)
    got = KeyedTensor.regroup([kt], [["dense_0", "dense_4"], ["dense_1", "dense_3"], ["dense_2"]])
    assert torch.equal(got[0], torch.cat([tensors[0], tensors[4]], 1))
    assert torch.equal(got[1], torch.cat([tensors[1], tensors[3]], 1))
    assert torch.equal(got[2], tensors[2])


@pytest.mark.parametrize("dev", DEVICES)
def test_regroup_multiple_kt_and_as_dict(dev):
    t1 = [torch.randn(2, 4, device=dev), torch.randn(2, 8, device=dev), torch.randn(2, 2, device=dev)]
    t2 = [torch.randn(2, 3, device=dev), torch.randn(2, 10, device=dev)]
    kt1 = KeyedTensor.from_tensor_list(["dense_0", "dense_1", "dense_2"], t1, 1)
    kt2 = KeyedTensor.from_tensor_list(["sparse_0", "sparse_1"], t2, 1)
    groups = [["dense_0", "sparse_1", "dense_2"], ["dense_1", "sparse_0"]]
    got = KeyedTensor.regroup([kt1, kt2], groups)
    assert torch.equal(got[0], torch.cat([t1[0], t2[1], t1[2]], 1))
    assert torch.equal(got[1], torch.cat([t1[1], t2[0]], 1))
    as_dict = KeyedTensor.regroup_as_dict([kt1, kt2], groups, ["a", "b"])
    assert list(as_dict) == ["a", "b"] and torch.equal(as_dict["b"], got[1])
    with pytest.raises(AssertionError):
        KeyedTensor.regroup_as_dict([kt1, kt2], groups, ["a"])


@pytest.mark.parametrize("dev", DEVICES)
def test_regroup_multiple_kt_duplicate_keys(dev):
    t1 = [torch.randn(2, 4, device=dev) for _ in range(2)]
    t2 = [torch.randn(2, 3, device=dev) for _ in range(3)]
    kt1 = KeyedTensor.from_tensor_list(["dense_0", "dense_1"], t1, 1)
    kt2 = KeyedTensor.from_tensor_list(["sparse_0", "sparse_1", "dense_2"], t2, 1)
    got = KeyedTensor.regroup([kt1, kt2], [["dense_0", "sparse_1"], ["dense_1", "sparse_0", "dense_0"]])
    assert torch.equal(got[0], torch.cat([t1[0], t2[1]], 1))
    assert torch.equal(got[1], torch.cat([t1[1], t2[0], t1[0]], 1))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_regroup_kernel_against_slicing(dtype):
    """Many keys (more than one launch's worth of blocks), odd widths, a key
    used twice, a key not used, an empty group."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(5)
    kts, all_keys = [], []
    for t in range(3):
        widths = rng.integers(1, 40, 70).tolist()
        keys = [f"k{t}_{i}" for i in range(len(widths))]
        values = torch.randn(257, sum(widths), device=dev).to(dtype)
        kts.append(KeyedTensor(keys=keys, length_per_key=widths, values=values))
        all_keys += keys
    order = rng.permutation(len(all_keys)).tolist()
    picked = [all_keys[i] for i in order[:-5]]  # five keys stay unused
    groups = [picked[:50], picked[50:51], [], picked[51:] + picked[:3]]
    want = _regroup_keyed_tensors(kts, groups)
    for fn in (regroup_kts, permute_multi_embedding, KeyedTensor.regroup):
        got = fn(kts, groups)
        assert len(got) == len(want)
        for g, w in zip(got, want):
            assert g.shape == w.shape and g.dtype == dtype and torch.equal(g, w)
    # a view with a row stride larger than its width (a slice of a wider output)
    wide = torch.randn(64, 100, device=dev).to(dtype)
    part = KeyedTensor(keys=["x", "y"], length_per_key=[30, 20], values=wide[:, 10:60])
    got = regroup_kts([part], [["y", "x"]])
    assert torch.equal(got[0], torch.cat([wide[:, 40:60], wide[:, 10:40]], 1))


@pytest.mark.gpu
@pytest.mark.parametrize("unit", [1, 2, 4, 8])  # fp16 columns per vector of 2, 4, 8, 16 bytes
@pytest.mark.parametrize("rows", [1, 3, 513, 2049, 16387])  # 1, 4 and 16 rows per thread, and remainders
def test_regroup_kernel_tiles(rows, unit):
    """Edges of the kernel's row and column tiles: one column vector, one more than a tile of 256."""
    dev = torch.device("cuda:0")
    for widths in ([unit], [unit * 256, unit], [unit * 40] * 13):
        keys = [f"k{i}" for i in range(len(widths))]
        # a pad column of one unit keeps the source rows aligned to the unit and no more
        wide = torch.randint(0, 2**15, (rows, sum(widths) + unit), device=dev, dtype=torch.int16).view(torch.float16)
        kt = KeyedTensor(keys=keys, length_per_key=widths, values=wide[:, unit:])
        groups = [keys[::-1], keys[:1]]
        for g, w in zip(regroup_kts([kt], groups), _regroup_keyed_tensors([kt], groups)):
            assert torch.equal(g.view(torch.int16), w.view(torch.int16))


@pytest.mark.parametrize("dev", DEVICES)
def test_kt_regroup_as_dict_module(dev):
    """torchrec/modules/tests/test_regroup.py: same result as the static method,
    on the first and on later batches; a duplicate key is refused; the cast."""
    from torchrec_amd.modules.embedding_configs import DataType
    from torchrec_amd.modules.regroup import KTRegroupAsDict

    def batch():
        t1 = [torch.randn(6, 4, device=dev), torch.randn(6, 8, device=dev), torch.randn(6, 2, device=dev)]
        t2 = [torch.randn(6, 3, device=dev), torch.randn(6, 10, device=dev)]
        return [KeyedTensor.from_tensor_list(["f1", "f2", "f3"], t1), KeyedTensor.from_tensor_list(["g1", "g2"], t2)]

    groups, keys = [["f1", "g2", "f3"], ["f2", "g1"]], ["object", "user"]
    m = KTRegroupAsDict(groups, keys)
    for _ in range(3):
        kts = batch()
        got, want = m(kts), KeyedTensor.regroup_as_dict(kts, groups, keys)
        assert list(got) == keys and all(torch.equal(got[k], want[k]) for k in keys)
    half = KTRegroupAsDict(groups, keys, emb_dtype=DataType.FP16)
    kts = batch()
    out = half(kts)
    assert out["user"].dtype == torch.float16
    assert torch.equal(out["user"], torch.cat([kts[0]["f2"], kts[1]["g1"]], 1).half())
    dup = [KeyedTensor.from_tensor_list(["f1"], [torch.randn(2, 2, device=dev)]),
           KeyedTensor.from_tensor_list(["f1"], [torch.randn(2, 2, device=dev)])]
    with pytest.raises(RuntimeError, match="Duplicate key"):
        KTRegroupAsDict([["f1"]], ["a"])(dup)
    m.clear_cache()
    assert not m._is_inited


@pytest.mark.parametrize("dev", DEVICES)
def test_regroup_module_saved_without_its_layout(dev):
    """A module that was saved after its first batch, before it kept the layout of its plan."""
    from torchrec_amd.modules.regroup import KTRegroupAsDict
    tensors = [torch.randn(3, 4, device=dev) for _ in range(3)]
    kt = KeyedTensor.from_tensor_list(["a", "b", "c"], tensors, 1)
    m = KTRegroupAsDict([["c", "a"], ["b"]], ["x", "y"])
    m([kt])
    del m.__dict__["_layout"]
    got = m([kt])
    assert torch.equal(got["x"], torch.cat([tensors[2], tensors[0]], 1)) and torch.equal(got["y"], tensors[1])


@pytest.mark.gpu
@pytest.mark.parametrize("elem,widths", [(2, [3, 8, 1]), (4, [5, 4, 64]), (4, [0, 7]), (2, [256] * 100)])
def test_regroup_columns_entry(elem, widths):
    """``tra_regroup_columns`` (blocks given by address): blocks in reverse order, in a wider row; bad blocks refused."""
    import ctypes

    from torchrec_amd import _lib
    dev, rows, total = torch.device("cuda:0"), 37, sum(widths)
    dtype = {2: torch.int16, 4: torch.int32}[elem]
    src = torch.randint(-30000, 30000, (rows, total + 3), device=dev).to(dtype)
    dst = torch.zeros(rows, total + 5, dtype=dtype, device=dev)
    n, at = len(widths), np.concatenate([[0], np.cumsum(widths)])
    to = total - at[1:]  # (the blocks from the right)
    vp, i64, i32 = ctypes.c_void_p * n, ctypes.c_int64 * n, ctypes.c_int32 * n
    args = [vp(*[src.data_ptr() + int(a) * elem for a in at[:-1]]), i64(*[total + 3] * n),
            vp(*[dst.data_ptr() + int(a) * elem for a in to]), i64(*[total + 5] * n), i32(*widths), n, rows, elem,
            _lib.current_stream(dev)]
    assert _lib.lib().tra_regroup_columns(*args) == 0
    want = torch.zeros_like(dst)
    for a, b, w in zip(at, to, widths):
        want[:, int(b):int(b) + w] = src[:, int(a):int(a) + w]
    assert torch.equal(dst, want)
    args[1] = i64(*[max(widths) - 1] * n)
    assert _lib.lib().tra_regroup_columns(*args) == -1
