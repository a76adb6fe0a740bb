"""The work that users of this package have it do, as cases that can be timed.

The package serves quantized embedding tables: a request arrives as a
KeyedJaggedTensor, is looked up (pooled per bag, or row by row), and leaves as
dense blocks.  Around that stand the conversion of a float model, the id
bucketization of row-wise sharding, the managed-collision remap and the
regrouping of pooled blocks.  ``listed()`` names twelve such calls, from the
smallest online request to the largest batch; ``draw(rng)`` gives others of the
same ranges.  Shapes are the ones of ``bench.py`` (its configurations c1 - c5)
or lie between them.

A case is a dict of plain values.  ``kind`` says which call it is:

* ``pooled``    quantized EmbeddingBagCollection (with ``position``: the
                feature-processed one), KJT -> KeyedTensor
* ``sequence``  quantized EmbeddingCollection (with ``collision``: behind a
                managed-collision remap), KJT -> one JaggedTensor per feature
* ``bucketize`` KJT -> KJT of ``buckets`` row-wise shards
* ``convert``   float EmbeddingBagCollection -> quantized one
* ``regroup``   KeyedTensors -> one dense block per group
"""
import math

import numpy as np
import torch
from torch.quantization import PlaceholderObserver

from torchrec_amd import KeyedJaggedTensor
from torchrec_amd.inference.modules import get_table_to_weights_from_tbe, quantize_inference_model
from torchrec_amd.modules.embedding_configs import (
    DataType,
    EmbeddingBagConfig,
    EmbeddingConfig,
    PoolingType,
    QuantConfig,
)
from torchrec_amd.modules.embedding_modules import EmbeddingBagCollection
from torchrec_amd.modules.feature_processor_ import PositionWeightedModuleCollection
from torchrec_amd.modules.mc_modules import ManagedCollisionCollection, MCHManagedCollisionModule
from torchrec_amd.modules.regroup import KTRegroupAsDict
from torchrec_amd.quant import EmbeddingBagCollection as QuantEmbeddingBagCollection
from torchrec_amd.quant import EmbeddingCollection as QuantEmbeddingCollection
from torchrec_amd.quant.embedding_modules import (
    FeatureProcessedEmbeddingBagCollection as QuantFeatureProcessedEmbeddingBagCollection,
    QuantManagedCollisionEmbeddingCollection,
    quant_prep_enable_register_tbes,
)
from torchrec_amd.sparse.bucketize import bucketize_kjt_inference
from torchrec_amd.sparse.jagged_tensor import KeyedTensor

_DATA_TYPES = {"int8": DataType.INT8, "int4": DataType.INT4, "int2": DataType.INT2, "fp16": DataType.FP16}
_BITS = {"int8": 8, "int4": 4, "int2": 2, "fp16": 16}
_QUANT_DTYPES = {"int8": torch.qint8, "int4": torch.quint4x2, "int2": torch.quint2x4}
_OUT = {"fp16": torch.half, "fp32": torch.float}
_INDEX = {"int32": torch.int32, "int64": torch.int64}

_POOLED = {
    "kind": "pooled", "features": 8, "batch": 512, "dims": "64", "types": "int8",
    "rows_lo": 100_000, "rows_hi": 100_000,  # rows of a table, log-uniform between the two
    "lengths": "fixed", "bag": 20, "empty": 0.0,  # fixed: bag; poisson: mean bag; uniform: 1 .. bag; share of empty bags
    "alpha": 0.0,  # ids: 0 uniform, else Zipf(alpha) over scattered rows
    "weighted": False, "position": False, "mean": False,
    "out": "fp16", "index": "int32",
    "given": "lengths",  # what the KJT was built from
    "shuffled": False,  # keys in another order than the tables' features, and one key that no table uses
    "row_alignment": 16,
    "converted": False,  # module made by quantize_inference_model from a float one
}
_SEQUENCE = {
    "kind": "sequence", "features": 16, "batch": 1024, "dims": "128", "types": "int8",
    "rows_lo": 1_000_000, "rows_hi": 1_000_000, "lengths": "uniform0", "bag": 256, "empty": 0.0, "alpha": 0.0,
    "out": "fp16", "index": "int32", "given": "lengths", "shuffled": False, "collision": False,
}
_BUCKETIZE = {
    "kind": "bucketize", "features": 64, "batch": 4096, "rows_lo": 100_000, "rows_hi": 10_000_000,
    "lengths": "poisson", "bag": 30, "empty": 0.0, "alpha": 0.0, "index": "int64", "given": "lengths",
    "weighted": True, "buckets": 8, "sequence": False,
}


def listed():
    return [
        # One online request scored against a handful of candidates: the whole call is latency.  The
        # module comes from the float model through quantize_inference_model, ids are torch's int64.
        dict(_POOLED, name="online", batch=16, lengths="poisson", out="fp32", index="int64", converted=True),
        # A small ranking batch (bench.py c1).
        dict(_POOLED, name="small"),
        # DLRM-style ranking, int4 tables, hot ids (bench.py c2).
        dict(_POOLED, name="dlrm", features=26, batch=2048, dims="128", types="int4", rows_lo=1000,
             rows_hi=40_000_000, lengths="uniform", bag=40, empty=0.05, alpha=1.05),
        # Mixed widths and weight types, per-sample weights, fp32 results (bench.py c3).
        dict(_POOLED, name="mixed", features=64, batch=4096, dims="32,64,128,256", types="int8,int4,int2,fp16",
             rows_lo=100_000, rows_hi=10_000_000, lengths="poisson", bag=30, weighted=True, out="fp32"),
        # Tables beyond the row-padding budget, long bags, MEAN (bench.py c5 with tables that fit three times).
        dict(_POOLED, name="large", features=8, batch=16384, dims="128", types="int4", rows_lo=70_000_000,
             rows_hi=70_000_000, bag=80, alpha=0.8, mean=True, row_alignment=4),
        # Position-weighted features of odd widths, an odd batch, keys as the data loader happens to order them.
        dict(_POOLED, name="position", features=20, batch=1531, dims="40,72,104", types="int8,int4", rows_lo=5_000,
             rows_hi=2_000_000, lengths="uniform", bag=50, empty=0.1, alpha=1.1, position=True, index="int64",
             shuffled=True),
        # User histories, row by row (bench.py c4).
        dict(_SEQUENCE, name="history"),
        # The same for a few users at once, int4 rows.
        dict(_SEQUENCE, name="history_online", features=4, batch=32, dims="64", types="int4", rows_lo=200_000,
             rows_hi=200_000, bag=50, index="int64"),
        # Raw 64-bit ids remapped through managed-collision tables, keys in another order than the tables.
        dict(_SEQUENCE, name="collision", features=8, batch=1024, dims="64", rows_lo=500_000, rows_hi=500_000,
             bag=100, alpha=1.05, index="int64", collision=True, shuffled=True),
        # The ids of row-wise shards: weighted features cut into 8 buckets (the bags of bench.py c3).
        dict(_BUCKETIZE, name="row_wise"),
        # A float collection becomes the served one.
        {"kind": "convert", "name": "convert", "features": 4, "dims": "128", "types": "int4", "rows_lo": 1_000_000,
         "rows_hi": 1_000_000},
        # Pooled blocks of three collections regrouped for the dense layers.
        {"kind": "regroup", "name": "regroup", "parts": 3, "features": 20, "dims": "32,64,128", "batch": 4096,
         "groups": 4, "out": "fp16"},
    ]


def _between(rng, lo, hi):
    """A whole number spread evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pooled"] * 6 + ["sequence"] * 3 + ["bucketize", "convert", "regroup"])
    index = rng.choice(["int32", "int64"])
    given = rng.choice(["lengths", "lengths", "offsets"])
    if kind == "pooled":
        features = _between(rng, 1, 64)
        bag = _between(rng, 1, 80)
        batch = max(1, _between(rng, 8, min(16384, 8_000_000 // (features * bag))))
        rows_hi = _between(rng, 1_000, min(40_000_000, 400_000_000 // features))
        extra = rng.choice(["none", "none", "weighted", "position"])
        return dict(
            _POOLED, features=features, batch=batch, bag=bag,
            dims=rng.choice(["64", "128", "32,64,128,256", "48,80,112", "16", "128,256"]),
            types=rng.choice(["int8", "int4", "int4", "int2", "fp16", "int8,int4,int2,fp16"]),
            rows_lo=_between(rng, 500, rows_hi) if rows_hi > 500 else rows_hi, rows_hi=rows_hi,
            lengths=rng.choice(["fixed", "poisson", "uniform"]), empty=rng.choice([0.0, 0.05, 0.3]),
            alpha=rng.choice([0.0, 0.8, 1.05, 1.2]), weighted=extra == "weighted", position=extra == "position",
            mean=extra != "position" and rng.random() < 0.25, out=rng.choice(["fp16", "fp16", "fp32"]), index=index,
            given=given, shuffled=rng.random() < 0.25, row_alignment=rng.choice([4, 16, 16]),
        )
    if kind == "sequence":
        features = _between(rng, 1, 26)
        bag = _between(rng, 2, 256)
        collision = rng.random() < 0.35
        return dict(
            _SEQUENCE, features=features, bag=bag,
            batch=max(1, _between(rng, 8, max(8, min(4096, (1_000_000 if collision else 4_000_000) // (features * bag))))),
            dims=rng.choice(["32", "64", "128", "104", "40"]), types=rng.choice(["int8", "int8", "int4", "fp16"]),
            rows_lo=1_000, rows_hi=_between(rng, 10_000, 1_000_000), lengths=rng.choice(["uniform0", "poisson", "fixed"]),
            alpha=rng.choice([0.0, 1.05]), out=rng.choice(["fp16", "fp32"]), index="int64" if collision else index,
            given=given, shuffled=rng.random() < 0.3, collision=collision,
        )
    if kind == "bucketize":
        features = _between(rng, 1, 64)
        bag = _between(rng, 1, 80)
        return dict(
            _BUCKETIZE, features=features, bag=bag, batch=_between(rng, 8, min(16384, 8_000_000 // (features * bag))),
            lengths=rng.choice(["poisson", "uniform"]), alpha=rng.choice([0.0, 1.05]), index=index, given=given,
            weighted=rng.random() < 0.5, buckets=rng.choice([2, 3, 4, 8, 16]), sequence=rng.random() < 0.5,
        )
    if kind == "convert":
        dims = rng.choice(["64", "128", "48,112", "32,64,128"])
        features = _between(rng, 1, 16)
        rows = _between(rng, 10_000, 3_500_000 // features)
        return {"kind": "convert", "features": features, "dims": dims,
                "types": rng.choice(["int8", "int4", "int2", "int8,int4"]), "rows_lo": rows // 2, "rows_hi": rows}
    return {"kind": "regroup", "parts": rng.randint(1, 4), "features": _between(rng, 2, 26),
            "dims": rng.choice(["64", "128", "32,64,128", "36,100"]), "batch": _between(rng, 16, 4096),
            "groups": rng.randint(1, 6), "out": rng.choice(["fp16", "fp32"])}


# --------------------------------------------------------------------------
# shapes shared by prepare() and work()
# --------------------------------------------------------------------------
def _tables(case):
    """[(rows, dim, type)] of the case's tables, one per feature; the same for every seed."""
    n = case["features"]
    dims = [int(d) for d in case.get("dims", "4").split(",")]
    types = case.get("types", "int8").split(",")
    rng = np.random.default_rng(n)
    lo, hi = math.log(case["rows_lo"]), math.log(case["rows_hi"])
    rows = [int(round(math.exp(x))) for x in rng.uniform(lo, hi, n)]
    # types change every time the dims have gone round, so that every width meets every type
    return [(max(rows[t], 2), dims[t % len(dims)], types[(t // len(dims)) % len(types)]) for t in range(n)]


def _row_bytes(dim, ty):
    return dim * _BITS[ty] // 8 + (0 if ty == "fp16" else 4)


def _ids_per_feature(case):
    mean = {"fixed": case["bag"], "poisson": case["bag"], "uniform": (case["bag"] + 1) / 2, "uniform0": case["bag"] / 2}
    return case["batch"] * mean[case["lengths"]] * (1.0 - case["empty"])


def _distinct(n, rows, alpha):
    """Expected distinct rows among n ids: a row that is met again need not be read again."""
    edges = np.exp(np.linspace(math.log(0.5), math.log(rows + 0.5), 257))
    if alpha:
        p = np.diff(edges ** (1.0 - alpha)) / (edges[-1] ** (1.0 - alpha) - edges[0] ** (1.0 - alpha))
    else:
        p = np.diff(edges) / rows
    width = np.diff(edges)
    return float(np.sum(width * -np.expm1(-n * p / width)))


def work(case):
    """Bytes of one pass: every id, length and weight once, every distinct row once (without padding), every
    result once.  ``flops``: two per pooled or dequantized element."""
    kind = case["kind"]
    if kind == "regroup":
        columns = sum(sum(part) for part in _parts(case))
        return {"bytes": 2 * case["batch"] * columns * (2 if case["out"] == "fp16" else 4), "flops": 0}
    tables = _tables(case)
    if kind == "convert":
        return {"bytes": sum(r * (4 * d + _row_bytes(d, ty)) for r, d, ty in tables),
                "flops": sum(2 * r * d for r, d, _ in tables)}
    n, isz, bags = _ids_per_feature(case), (4 if case["index"] == "int32" else 8), case["features"] * case["batch"]
    ids = n * case["features"]
    if kind == "bucketize":
        per_id = 2 * (isz + (4 if case["weighted"] else 0)) + (8 + isz if case["sequence"] else 0)
        return {"bytes": ids * per_id + bags * isz * (1 + case["buckets"]), "flops": 0}
    osz = 2 if case["out"] == "fp16" else 4
    moved = ids * (isz + (4 if case.get("weighted") else 0)) + bags * isz
    moved += sum(_distinct(n, r, case["alpha"]) * _row_bytes(d, ty) for r, d, ty in tables)
    if kind == "sequence":
        moved += sum(n * d * osz for _, d, _ in tables)
        if case["collision"]:  # the remapped ids are a result; a known id's table entry and row are read
            moved += ids * isz + sum(_distinct(n, r, case["alpha"]) * 16 for r, _, _ in tables)
    else:
        moved += case["batch"] * sum(d for _, d, _ in tables) * osz
    return {"bytes": moved, "flops": sum(2 * n * d for _, d, _ in tables)}


def tolerance(case):
    """Bytes and whole numbers are the same.  Looked-up values: against the same sums in 64 bits, fp32 results are
    off by 2.5e-7 (largest 8e-7) at 80 ids a bag, fp16 results by their own rounding, 2.1e-4 (largest 4.9e-4)."""
    if case["kind"] in ("bucketize", "convert", "regroup"):
        return "exact"
    return {"rel": 8e-4, "max": 2e-3} if case["out"] == "fp16" else {"rel": 1e-6, "max": 4e-6}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _fill(module, gen):
    """Random rows in the packed tables of a quantized module: any payload, plausible scale and bias."""
    for op in module._emb_modules:
        for payload, scale, bias in op.split_embedding_weights_with_scale_bias(2):
            if scale is None:
                payload.view(torch.float16).normal_(0, 0.1, generator=gen)
            else:
                payload.view(torch.int32).random_(-(2**31), 2**31 - 1, generator=gen)
                scale.uniform_(0.004, 0.02, generator=gen)
                bias.uniform_(-0.15, -0.03, generator=gen)


def _lengths(case, keys, gen):
    """Lengths [keys * batch].  A key's lengths are the same for every seed, in another order: jagged results then
    have the same number of rows whatever the ids."""
    bag, how, shape = case["bag"], case["lengths"], (keys, case["batch"])
    fixed = _generator(1)
    if how == "fixed":
        lengths = torch.full(shape, bag, device="cuda")
    elif how == "poisson":
        lengths = torch.poisson(torch.full(shape, float(bag), device="cuda"), generator=fixed).long()
    else:
        lengths = torch.randint(1 if how == "uniform" else 0, bag + 1, shape, device="cuda", generator=fixed)
    if case["empty"]:
        lengths *= torch.rand(shape, device="cuda", generator=fixed) >= case["empty"]
    order = torch.rand(shape, device="cuda", generator=gen).argsort(dim=1)
    return lengths.gather(1, order).view(-1)


def _draw_ids(n, rows, alpha, gen):
    """n ids of [0, rows): uniform, or Zipf(alpha) ranks scattered over the table."""
    if not alpha:
        return torch.randint(0, rows, (n,), device="cuda", generator=gen)
    a, lo = 1.0 - alpha, 0.5
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    rank = (u * ((rows + lo) ** a - lo**a) + lo**a).pow_(1.0 / a).add_(0.5).long().sub_(1).clamp_(0, rows - 1)
    mul = 2654435761 % rows or 1
    while math.gcd(mul, rows) != 1:
        mul += 1
    return (rank * mul + 12345) % rows


def _request(case, keys, rows, gen, weighted=False, id_tables=None):
    """(keys, values, lengths, offsets, weights) of a request: ids of key i lie in [0, rows[i]).  ``id_tables``:
    raw ids by table row; one id in ten is one that no table knows."""
    lengths = _lengths(case, len(keys), gen)
    per_key = lengths.view(len(keys), -1).sum(1).tolist()
    parts = []
    for key, n, r in zip(keys, per_key, rows):
        ids = _draw_ids(n, r, case["alpha"], gen)
        if id_tables is not None:
            raw = id_tables[key]
            unknown = torch.randint(0, 2**40, (n,), device="cuda", generator=gen)
            ids = torch.where(torch.rand(n, device="cuda", generator=gen) < 0.9, raw[ids % raw.numel()], unknown)
        parts.append(ids)
    dtype = _INDEX[case["index"]]
    values = torch.cat(parts).to(dtype)
    lengths = lengths.to(dtype)
    offsets = None
    if case["given"] == "offsets":
        offsets = torch.zeros(lengths.numel() + 1, dtype=dtype, device="cuda")
        offsets[1:] = torch.cumsum(lengths, 0)
        lengths = None
    weights = torch.rand(values.numel(), device="cuda", generator=gen) if weighted else None
    return {"keys": keys, "values": values, "lengths": lengths, "offsets": offsets, "weights": weights}


def _key_order(case, rows):
    """(keys, rows per key): the features in order, or shuffled with a key among them that no table uses."""
    keys = ["f%d" % i for i in range(len(rows))]
    if not case.get("shuffled"):
        return keys, rows
    if not case.get("collision"):  # (a managed-collision collection takes its own features only)
        keys, rows = keys + ["unused"], rows + [1000]
    order = np.random.default_rng(len(rows)).permutation(len(keys))
    return [keys[i] for i in order], [rows[i] for i in order]


def _configs(case, config_type, **more):
    return [
        config_type(name="t%d" % i, embedding_dim=d, num_embeddings=r, feature_names=["f%d" % i],
                    data_type=_DATA_TYPES[ty], **more)
        for i, (r, d, ty) in enumerate(_tables(case))
    ]


def _float_collection(case, gen):
    tables = [
        EmbeddingBagConfig(name="t%d" % i, embedding_dim=d, num_embeddings=r, feature_names=["f%d" % i])
        for i, (r, d, _) in enumerate(_tables(case))
    ]
    module = EmbeddingBagCollection(tables, device=torch.device("cuda", 0))
    with torch.no_grad():
        for p in module.parameters():
            p.normal_(0, 0.1, generator=gen)
    return module


def _prepare_pooled(case, gen):
    device = torch.device("cuda", 0)
    specs = _tables(case)
    if case["converted"]:
        model = torch.nn.Sequential(_float_collection(case, gen))
        module = quantize_inference_model(model, quantization_dtype=_QUANT_DTYPES[case["types"]],
                                          output_dtype=_OUT[case["out"]])[0]
    else:
        tables = _configs(case, EmbeddingBagConfig, pooling=PoolingType.MEAN if case["mean"] else PoolingType.SUM)
        more = {"output_dtype": _OUT[case["out"]], "row_alignment": case["row_alignment"]}
        if case["position"]:
            # every third feature is pooled without position weights
            spans = {"f%d" % i: case["bag"] for i in range(len(specs)) if i % 3 != 2}
            processor = PositionWeightedModuleCollection(spans, device=device)
            with torch.no_grad():
                for p in processor.position_weights.values():
                    p.uniform_(0.1, 1.0, generator=gen)
            module = QuantFeatureProcessedEmbeddingBagCollection(tables, True, device, feature_processor=processor, **more)
        else:
            module = QuantEmbeddingBagCollection(tables, case["weighted"], device, **more)
        _fill(module, gen)
    keys, rows = _key_order(case, [r for r, _, _ in specs])
    return {"module": module, "request": _request(case, keys, rows, gen, case["weighted"])}


def _prepare_sequence(case, gen):
    device = torch.device("cuda", 0)
    specs = _tables(case)
    tables = _configs(case, EmbeddingConfig)
    keys, rows = _key_order(case, [r for r, _, _ in specs])
    id_tables = None
    if case["collision"]:
        managed, id_tables = {}, {}
        for table, (r, _, _) in zip(tables, specs):
            raw = torch.unique(torch.randint(0, 2**40, (r - 1,), device=device, generator=gen))
            raw = raw[torch.randperm(raw.numel(), device=device, generator=gen)]
            managed[table.name] = MCHManagedCollisionModule(r, device)
            managed[table.name].set_id_table(raw, torch.randperm(r - 1, device=device, generator=gen)[: raw.numel()])
            id_tables[table.feature_names[0]] = raw
        module = QuantManagedCollisionEmbeddingCollection(
            tables, device, output_dtype=_OUT[case["out"]],
            managed_collision_collection=ManagedCollisionCollection(managed, tables),
        )
    else:
        module = QuantEmbeddingCollection(tables, device, output_dtype=_OUT[case["out"]])
    _fill(module, gen)
    return {"module": module, "request": _request(case, keys, rows, gen, False, id_tables)}


def _prepare_bucketize(case, gen):
    rows = [r for r, _, _ in _tables(case)]
    keys = ["f%d" % i for i in range(len(rows))]
    w = case["buckets"]
    block_sizes = torch.tensor([-(-r // w) for r in rows], dtype=torch.int64, device="cuda")
    return {"block_sizes": block_sizes, "request": _request(case, keys, rows, gen, case["weighted"])}


def _prepare_convert(case, gen):
    module = _float_collection(case, gen)
    per_table = {"t%d" % i: _QUANT_DTYPES[ty] for i, (_, _, ty) in enumerate(_tables(case))}
    module.qconfig = QuantConfig(
        activation=PlaceholderObserver.with_args(dtype=torch.half),
        weight=PlaceholderObserver.with_args(dtype=per_table["t0"]), per_table_weight_dtype=per_table,
    )
    quant_prep_enable_register_tbes(module, [EmbeddingBagCollection])
    return {"module": module}


def _parts(case):
    """Block widths of every KeyedTensor."""
    dims = [int(d) for d in case["dims"].split(",")]
    return [[dims[(p + i) % len(dims)] for i in range(case["features"])] for p in range(case["parts"])]


def _prepare_regroup(case, gen):
    parts, names = [], []
    for p, widths in enumerate(_parts(case)):
        keys = ["p%d_f%d" % (p, i) for i in range(len(widths))]
        values = torch.empty(case["batch"], sum(widths), dtype=_OUT[case["out"]], device="cuda")
        values.normal_(generator=gen)
        parts.append((keys, widths, values))
        names += keys
    order = np.random.default_rng(len(names)).permutation(len(names))
    groups = [[names[i] for i in order[g :: case["groups"]]] for g in range(case["groups"])]
    return {"module": KTRegroupAsDict(groups, ["g%d" % g for g in range(len(groups))]), "parts": parts}


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "pooled":
        state = _prepare_pooled(case, gen)
    elif kind == "sequence":
        state = _prepare_sequence(case, gen)
    elif kind == "bucketize":
        state = _prepare_bucketize(case, gen)
    elif kind == "convert":
        state = _prepare_convert(case, gen)
    else:
        state = _prepare_regroup(case, gen)
    state["case"] = case
    return state


# --------------------------------------------------------------------------
# the calls
# --------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "convert":
        quantized = QuantEmbeddingBagCollection.from_float(state["module"])
        return get_table_to_weights_from_tbe(quantized)
    if kind == "regroup":
        return state["module"]([KeyedTensor(keys=k, length_per_key=w, values=v) for k, w, v in state["parts"]])
    kjt = KeyedJaggedTensor(**state["request"])
    if kind == "pooled":
        return state["module"](kjt).values()
    if kind == "bucketize":
        out, order, bucket = bucketize_kjt_inference(
            kjt, case["buckets"], state["block_sizes"], is_sequence=case["sequence"]
        )
        return {"values": out.values(), "lengths": out.lengths(), "weights": out.weights_or_none(), "order": order,
                "bucket": bucket}
    if case["collision"]:
        found, remapped = state["module"](kjt)
        return {"rows": {k: jt.values() for k, jt in found.items()}, "ids": remapped.values()}
    return {k: jt.values() for k, jt in state["module"](kjt).items()}
