"""The sixteen-lane pooled kernel (calls too small for the window kernel) at the sizes where its lane groups, blocks of
sixteen ids and column slices begin and end, against the CPU oracle, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_equal, make_table
from test_tbe_gpu import DEV, build, _from_lengths, _launch_text
from torchrec_amd import _lib

pytestmark = pytest.mark.gpu

# one lane's columns change at 16, 32, 64, 128 and 256; 100 (int8) and 200 (int4) go by 32 lanes, 264 (int4) by 64;
# 300 and 520 (int8), 130 (fp16), 65 (fp32) are several slices
DIMS = {O.INT8: [4, 16, 20, 32, 64, 72, 100, 128, 256, 300, 520], O.INT4: [8, 16, 40, 64, 104, 128, 200, 256, 264],
        O.INT2: [16, 32, 64, 80, 256, 272], O.FP16: [2, 16, 18, 64, 66, 128, 130, 256], O.FP32: [1, 16, 17, 33, 64, 65, 128]}


def _lengths(rng, n):
    return rng.choice([0, 0, 1, 2, 7, 8, 9, 15, 16, 17, 31, 33, 70], n)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("dtype", [O.INT8, O.INT4, O.INT2, O.FP16, O.FP32])
def test_group_widths(tuning, dtype, weighted):
    tuning(balanced=0)
    rng = np.random.default_rng(70 + dtype * 2 + weighted)
    specs = [(dtype, 200 + 3 * i, dim) for i, dim in enumerate(DIMS[dtype])]
    ftm = list(range(len(specs)))
    idt, pooling, out = (np.int64, O.MEAN, O.FP32) if weighted else (np.int32, O.SUM, O.FP16)
    tbe, store = build(rng, specs, ftm, pooling, out, 4)
    for B in (1, 17, 65):
        lengths = _lengths(rng, len(specs) * B).astype(idt)
        offsets = np.zeros(len(lengths) + 1, dtype=idt)
        offsets[1:] = np.cumsum(lengths)
        per = lengths.reshape(len(specs), B).sum(1)
        ids = np.concatenate([rng.integers(-1, s[1], n) for s, n in zip(specs, per)]).astype(idt)
        psw = rng.uniform(-1, 1, len(ids)).astype(np.float32) if weighted else None
        want = O.tbe_forward(store, ftm, B, ids, offsets, psw, pooling, out)
        got = _from_lengths(tbe, ids, lengths, psw, B)
        assert bits_equal(got, want) == 0, B
        got = tbe(torch.from_numpy(ids).to(DEV), torch.from_numpy(offsets).to(DEV),
                  None if psw is None else torch.from_numpy(psw).to(DEV)).cpu().numpy()
        assert bits_equal(got, want) == 0, B


# 32 and 64 lanes a bag, and what 64 cannot hold (int8 of 144 and 256: 32 where bags are few, else 16)
WIDE = {O.INT8: [100, 144, 256, 260, 264, 300, 504, 512, 1020, 1024, 1040], O.INT4: [264, 512, 520, 1024, 1032],
        O.INT2: [272, 512, 1024, 1040], O.FP16: [130, 136, 256, 258, 512, 522], O.FP32: [65, 68, 128, 130, 256, 259, 516]}


@pytest.mark.parametrize("weights", ["none", "sample", "position"])
@pytest.mark.parametrize("dtype", list(WIDE))
def test_rows_of_more_than_sixteen_lanes(tuning, dtype, weights):
    tuning(balanced=0)
    rng = np.random.default_rng(dtype * 3 + len(weights))
    rows, T = 120, len(WIDE[dtype])
    idt, pooling, out = {"none": (np.int32, O.SUM, O.FP16), "sample": (np.int64, O.MEAN, O.FP32),
                         "position": (np.int32, O.SUM, O.FP32)}[weights]
    tbe, store = build(rng, [(dtype, rows, dim) for dim in WIDE[dtype]], list(range(T)), pooling, out, 4)
    bad = 0
    for B in (1, 9, 2000 if weights == "none" else 40):  # (2000: several bags per lane group)
        lengths = (rng.integers(0, 4, T * B) if B == 2000 else _lengths(rng, T * B)).astype(idt)
        offsets = np.zeros(T * B + 1, dtype=idt)
        offsets[1:] = np.cumsum(lengths)
        ids = rng.integers(-2, rows + 1, int(offsets[-1])).astype(idt)
        outside = (ids < -1) | (ids >= rows)
        psw, kw = None, {}
        if weights == "sample":
            psw = rng.uniform(-1, 1, len(ids)).astype(np.float32)
        elif weights == "position":
            table = rng.uniform(-1, 1, 6 * T).astype(np.float32)
            place, key = np.arange(len(ids)) - np.repeat(offsets[:-1], lengths), np.repeat(np.arange(T * B) // B, lengths)
            w = table[6 * key + np.minimum(place, 5)]
            kw = {"position_weights": (torch.from_numpy(table).to(DEV), [6 * t for t in range(T)], [6] * T)}
        want = O.tbe_forward(store, list(range(T)), B, np.where(outside, -1, ids).astype(idt), offsets,
                             w if weights == "position" else psw, pooling, out)
        got = _from_lengths(tbe, ids, lengths, psw, B, **kw)
        assert bits_equal(got, want) == 0, B
        got = tbe(torch.from_numpy(ids).to(DEV), torch.from_numpy(offsets).to(DEV),
                  None if psw is None else torch.from_numpy(psw).to(DEV), **kw).cpu().numpy()
        assert bits_equal(got, want) == 0, B
        bad += 2 * int(outside.sum())
    assert tbe.out_of_range_count() == bad


@pytest.mark.parametrize("bags", [40_000, 300_000])  # 3 and 16 bags per group
def test_several_bags_per_group(tuning, bags):
    tuning(balanced=0)
    rng = np.random.default_rng(bags)
    specs, B = [(O.INT8, 300, 16), (O.INT4, 200, 40)], bags // 2
    tbe, store = build(rng, specs, [0, 1], O.MEAN, O.FP32, 16)
    lengths = rng.choice([0, 1, 2, 17], 2 * B, p=[0.4, 0.3, 0.28, 0.02]).astype(np.int32)
    offsets = np.zeros(2 * B + 1, dtype=np.int32)
    offsets[1:] = np.cumsum(lengths)
    ids = rng.integers(0, 200, int(offsets[-1])).astype(np.int32)
    want = O.tbe_forward(store, [0, 1], B, ids, offsets, None, O.MEAN, O.FP32)
    assert bits_equal(_from_lengths(tbe, ids, lengths, None, B), want) == 0


@pytest.mark.parametrize("route", ["lengths", "scan", "offsets"])
@pytest.mark.parametrize("T,B,dim", [(1, 1000, 16), (1, 16_000, 100), (2, 40_000, 16)])  # 1, 2 and 5 bags per group
def test_counts_beyond_32_bits(tuning, T, B, dim, route):
    """Malformed 64-bit lengths and the offsets that they sum to: a count is cut to 32 bits, its bag is empty if that
    is negative, positions outside the ids read the last one; every other bag is pooled from its own bounds."""
    tuning(balanced=0)
    if route == "scan":
        tuning(fused_scan=0)
    rng = np.random.default_rng(T)
    tbe, store = build(rng, [(O.INT8, 300 + t, dim) for t in range(T)], list(range(T)), O.SUM, O.FP32, 16)
    lengths = rng.integers(0, 4, T * B).astype(np.int64)
    odd = rng.choice(T * B - 40, 200, replace=False)
    for k, x in enumerate((2**32 + 3, -(2**32) + 2, 2**40, -(2**40), 2**31 + 9, -(2**32) - 6, -5, 2**33 + 1)):
        lengths[odd[k::8]] = x
    lengths[0] = 3
    offsets = np.concatenate([[0], np.cumsum(lengths)])
    ids = rng.integers(0, 300, int(lengths[(lengths > 0) & (lengths < 4)].sum())).astype(np.int64)
    cut = lengths.astype(np.int32).clip(min=0).astype(np.int64)
    assert cut.max() < 4
    place = np.arange(int(cut.sum())) - np.repeat(np.cumsum(cut) - cut, cut)
    at = np.repeat(offsets[:-1], cut) + place
    at = np.where((at >= 0) & (at < len(ids)), at, len(ids) - 1)
    want = O.tbe_forward(store, list(range(T)), B, ids[at], np.concatenate([[0], np.cumsum(cut)]), None, O.SUM, O.FP32)
    ti = torch.from_numpy(ids).to(DEV)
    if route == "offsets":
        got = tbe(ti, torch.from_numpy(offsets).to(DEV), batch_size=B)
    else:
        got = tbe(ti, None, lengths=torch.from_numpy(lengths).to(DEV), batch_size=B)
    assert bits_equal(got.cpu().numpy(), want) == 0


def test_position_weights_of_many_slices():
    """150 features of two weight types: more than the launch arguments describe at once, no class above the limit."""
    rng = np.random.default_rng(5)
    T, B = 150, 5
    specs = [((O.INT8, O.INT4)[t % 2], 50, 16) for t in range(T)]
    tbe, store = build(rng, specs, list(range(T)), O.SUM, O.FP32, 16)
    lengths = rng.integers(0, 6, T * B).astype(np.int32)
    offsets = np.zeros(T * B + 1, dtype=np.int32)
    offsets[1:] = np.cumsum(lengths)
    ids = rng.integers(0, 50, int(offsets[-1])).astype(np.int32)
    table = rng.uniform(-1, 1, 4 * T).astype(np.float32)
    start, n = [4 * t for t in range(T)], [4 if t % 3 else 0 for t in range(T)]
    place = np.arange(len(ids)) - np.repeat(offsets[:-1], lengths)
    key = np.repeat(np.arange(T * B) // B, lengths)
    psw = np.where(np.take(n, key) > 0, table[np.take(start, key) + np.minimum(place, 3)], 1.0).astype(np.float32)
    want = O.tbe_forward(store, list(range(T)), B, ids, offsets, psw, O.SUM, O.FP32)
    got = tbe(torch.from_numpy(ids).to(DEV), torch.from_numpy(offsets).to(DEV),
              position_weights=(torch.from_numpy(table).to(DEV), start, n)).cpu().numpy()
    assert bits_equal(got, want) == 0


@pytest.mark.parametrize("dtype,dim", [(O.INT8, 64), (O.INT4, 128), (O.INT2, 256), (O.FP16, 64), (O.INT8, 300)])
def test_table_beyond_four_gib(tuning, dtype, dim):
    """Rows 4 MiB apart, 1100 of them: offsets beyond 32 bits.  The same rows close together give the same bits."""
    tuning(balanced=0)
    rng = np.random.default_rng(dim)
    rows, B = 1100, 33
    data = make_table(rng, dtype, rows, dim)
    if dtype not in (O.FP16, O.FP32):
        data = np.concatenate([data[:, -4:], data[:, :-4]], 1)  # (the operator's rows have the header in front)
    data = torch.from_numpy(np.ascontiguousarray(data).view(np.uint8).reshape(rows, -1)).to(DEV)
    lengths = _lengths(rng, B)
    offsets = torch.zeros(B + 1, dtype=torch.int32, device=DEV)
    offsets[1:] = torch.from_numpy(np.cumsum(lengths)).to(DEV)
    ids = torch.from_numpy(rng.integers(0, rows, int(lengths.sum())).astype(np.int32)).to(DEV)
    outs = []
    for stride in (data.shape[1], 4 << 20):
        store = torch.empty(rows * stride, dtype=torch.uint8, device=DEV)
        store.view(rows, stride)[:, : data.shape[1]].copy_(data)
        spec = (_lib.TableSpec * 1)()
        spec[0].offset, spec[0].rows, spec[0].dim, spec[0].row_bytes = 0, rows, dim, stride
        spec[0].dtype = {O.INT8: _lib.INT8, O.INT4: _lib.INT4, O.INT2: _lib.INT2, O.FP16: _lib.FP16}[dtype]
        plan = ctypes.c_void_p()
        l = _lib.lib()
        _lib.check(l.tra_tbe_create(spec, 1, (ctypes.c_int32 * 1)(0), None, 1, ctypes.byref(plan)))
        out = torch.empty(B, dim, device=DEV)
        _lib.check(l.tra_tbe_forward(plan, _lib.ptr(store), _lib.ptr(ids), _lib.ptr(offsets), 0, None, B, ids.numel(),
                                     _lib.POOL_SUM, _lib.FP32, _lib.ptr(out), dim, _lib.current_stream(DEV)))
        torch.cuda.synchronize()
        _lib.check(l.tra_tbe_destroy(plan))
        outs.append(out)
    assert outs[0].abs().max() > 0 and torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("idt", [np.int32, np.int64])
def test_one_class_line_to_the_window_kernel(idt, weighted):
    """One launch class: the sixteen-lane kernel up to 40 bags per compute unit, rows of whole bytes in bags of 8 ids and
    more up to 32; where a window would span more features than it can derive starts for, one launch of the
    sixteen-lane kernel up to 16,384 lengths of few ids.  Both sides of each line against the oracle."""
    rng = np.random.default_rng(77 + weighted)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    few, some = [0, 1, 2, 7], [9, 10]
    for dtype, T, B, lens, kernel in (
            (O.INT8, 8, 4 * cus, some, "tbe_pooled_kernel"), (O.INT8, 8, 4 * cus + 1, some, "tbe_pooled_cu_kernel"),
            (O.INT8, 8, 4 * cus + 1, few, "tbe_pooled_kernel"), (O.INT4, 8, 4 * cus + 1, some, "tbe_pooled_kernel"),
            (O.INT8, 8, 5 * cus, few, "tbe_pooled_cu_kernel"), (O.INT8, 200, 52, few, "tbe_pooled_kernel"),
            (O.INT8, 240, 66, few, "tbe_pooled_kernel"), (O.INT8, 249, 66, few, "tbe_pooled_cu_kernel"),
            (O.FP16, 128, 67, some, "tbe_pooled_cu_kernel")):
        tbe, store = build(rng, [(dtype, 40, 16)] * T, list(range(T)), O.SUM, O.FP32, 16)
        lengths = rng.choice(lens, T * B).astype(idt)
        offsets = np.zeros(T * B + 1, dtype=idt)
        offsets[1:] = np.cumsum(lengths)
        ids = rng.integers(0, 40, int(offsets[-1])).astype(idt)
        psw = rng.uniform(-1, 1, len(ids)).astype(np.float32) if weighted else None
        text = _launch_text(tbe, B, len(ids), T)
        assert kernel in text and ("scan" not in text) == (T * B <= 16384), (T, B, text)
        want = O.tbe_forward(store, list(range(T)), B, ids, offsets, psw, O.SUM, O.FP32)
        assert bits_equal(_from_lengths(tbe, ids, lengths, psw, B), want) == 0, (T, B)


@pytest.mark.parametrize("T", [64, 65])
def test_few_bags_take_one_launch_of_position_weights(T):
    """int8 rows of 256 columns go by 32 lanes, two descriptors each, where bags are few, but not beyond the 128 that a
    launch describes position weights for."""
    rng = np.random.default_rng(T)
    tbe, store = build(rng, [(O.INT8, 20, 256)] * T, list(range(T)), O.SUM, O.FP32, 16)
    B = 3
    assert f"slices={128 if T == 64 else T}" in _launch_text(tbe, B, 10, T)
    lengths = rng.integers(0, 4, T * B).astype(np.int32)
    offsets = np.zeros(T * B + 1, dtype=np.int32)
    offsets[1:] = np.cumsum(lengths)
    ids = rng.integers(0, 20, int(offsets[-1])).astype(np.int32)
    table = rng.uniform(-1, 1, 6 * T).astype(np.float32)
    place, key = np.arange(len(ids)) - np.repeat(offsets[:-1], lengths), np.repeat(np.arange(T * B) // B, lengths)
    want = O.tbe_forward(store, list(range(T)), B, ids, offsets, table[6 * key + place], O.SUM, O.FP32)
    pw = (torch.from_numpy(table).to(DEV), [6 * t for t in range(T)], [6] * T)
    assert bits_equal(_from_lengths(tbe, ids, lengths, None, B, position_weights=pw), want) == 0
