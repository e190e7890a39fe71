"""Performance cases: the work users of this package run, through its public entry points.

Four kinds of call, each over the range it is used in:

  pooled      IntNBitTableBatchedEmbeddingBagsCodegen.forward with SUM / MEAN pooling
  nobag       the same module with pooling_mode NONE (sequence embeddings)
  permute     PermutePooledEmbeddings forward and backward
  bucketize   torch.ops.fbgemm.block_bucketize_sparse_features

A case is a dict of plain values.  listed() gives the named cases, draw(rng) one more
case of the same ranges.  Index popularity is Zipf with the ranks scattered over the
table, as in the benchmark's configurations; INT rows hold codes of a min-max
quantised table, float rows normal values.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from __graft_entry__ import load_package

BITS = {"fp32": 32, "fp16": 16, "bf16": 16, "fp8": 8, "int8": 8, "int4": 4, "int2": 2}
TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16,
         "int32": torch.int32, "int64": torch.int64}
INT_ROWS = ("int8", "int4", "int2")


def _tbe(name, **kw):
    base = dict(name=name, kind="pooled", tables=1, rows_lo=100_000, rows_hi=100_000, dims="128", types="int8",
                layout=0, batch=512, bags="fixed:20", zipf=1.05, tail=0.0, index="int32", mode="sum", out="fp16",
                weighted=False)
    base.update(kw)
    return base


def listed():
    return [
        # a few quantised tables and a small batch: what one online ranking request costs
        _tbe("pooled_small", tables=8, zipf=0.0, index="int64", out="fp32"),
        # the 64 mixed tables of a ranking model at an online batch: many table groups, few bags
        _tbe("pooled_mixed_online", tables=64, rows_lo=10_000, rows_hi=500_000, dims="32,64,128,256",
             types="fp16:1,int8:3,int4:4,int2:2", layout=3, batch=32, bags="uniform:0:64", zipf=1.1, mode="mean",
             out="fp32", weighted=True),
        # FP8 tables of ragged widths, weighted, bf16 out: the reference's own test shapes at a ranking batch
        _tbe("pooled_fp8_ragged", tables=10, rows_lo=1_000, rows_hi=20_000, dims="ragged:4:1024", types="fp8:1",
             layout=8, batch=512, bags="uniform:1:100", zipf=0.0, index="int64", out="bf16", weighted=True),
        # unquantised tables with long rows (float models served as they were trained)
        _tbe("pooled_float_rows", tables=12, rows_lo=100_000, rows_hi=500_000, dims="64,128,256,512",
             types="bf16:2,fp32:1", layout=5, batch=2048, bags="poisson:30:1:100", out="bf16"),
        # 26 INT4 tables at a batch-inference size, the shape the headline number is quoted on
        _tbe("pooled_int4", tables=26, rows_lo=4_000_000, rows_hi=4_000_000, types="int4:1", batch=8192,
             bags="poisson:30:1:100"),
        # 64 mixed tables, weighted mean, at the full batch
        _tbe("pooled_mixed", tables=64, rows_lo=100_000, rows_hi=5_000_000, dims="32,64,128,256",
             types="fp16:1,int8:3,int4:4,int2:2", layout=3, batch=16384, bags="uniform:0:64", zipf=1.1, mode="mean",
             out="fp32", weighted=True),
        # 200 INT4 tables, int64 indices with a uniform tail: the largest pooled call (rows cut to fit three states)
        _tbe("pooled_int4_many", tables=200, rows_lo=1_000_000, rows_hi=1_000_000, types="int4:1", batch=8192,
             bags="poisson:40:1:128", zipf=1.2, tail=0.05, index="int64"),
        # sequence embeddings of 26 quantised tables: one output row per index
        _tbe("nobag_int8", kind="nobag", tables=26, rows_lo=1_000_000, rows_hi=1_000_000, types="int8:1",
             batch=2048, bags="poisson:30:1:100", mode="none"),
        # reorder of a pooled output of ragged features, with its backward (training of the dense part)
        dict(name="permute_ragged", kind="permute", features=64, dims="8,20,32,64,100,128,256", layout=4, batch=8192,
             out="fp16"),
        # a small weighted sequence batch split over 12 ranks: launches and latency
        dict(name="bucketize_small", kind="bucketize", features=48, batch=32, lengths="uniform:8:40", blocks="16:24",
             ranks=12, index="int64", weighted=True, positions=False, sequence=True, bucket_pos=True),
        # uneven row shards (bucket boundaries given per feature), weighted sequences
        dict(name="bucketize_uneven", kind="bucketize", features=96, batch=128, lengths="uniform:32:128",
             blocks="10000:1000000", ranks=8, index="int32", weighted=True, positions=True, sequence=True,
             bucket_pos=False),
        # the largest input redistribution: 42 M int64 indices to 16 ranks
        dict(name="bucketize_stress", kind="bucketize", features=16, batch=8192, lengths="uniform:128:512",
             blocks="128:256", ranks=16, index="int64", weighted=False, positions=False, sequence=False,
             bucket_pos=False),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pooled", "pooled", "pooled", "nobag", "permute", "bucketize", "bucketize"])
    if kind == "permute":
        features, batch = _logint(rng, 2, 200), _logint(rng, 16, 16384)
        dims = rng.choice(["8,20,32,64,100,128,256", "64,128", "128", "4,12,36,60", "1,3,5,16,31", "256,512"])
        while features * batch * max(map(int, dims.split(","))) > 4e8:
            batch = batch // 2
        return dict(kind=kind, features=features, dims=dims, layout=rng.randrange(1000), batch=batch,
                    out=rng.choice(["fp32", "fp16", "bf16"]))
    if kind == "bucketize":
        features, batch, mean = _logint(rng, 1, 100), _logint(rng, 1, 8192), _logint(rng, 2, 320)
        while features * batch * mean > 2e7:
            batch = batch // 2
        lo, ranks = _logint(rng, 8, 100_000), rng.choice([1, 2, 3, 5, 6, 8, 12, 16, 24, 32, 64, 128])
        while features * batch * ranks > 2e7:
            batch = batch // 2
        return dict(kind=kind, features=features, batch=max(1, batch), lengths=f"uniform:{mean // 2}:{mean * 3 // 2}",
                    blocks=f"{lo}:{2 * lo}", ranks=ranks, index=rng.choice(["int32", "int64"]),
                    weighted=rng.random() < 0.4, positions=rng.random() < 0.25, sequence=rng.random() < 0.5,
                    bucket_pos=rng.random() < 0.3)
    tables, batch, mean = _logint(rng, 1, 200), _logint(rng, 1, 8192), _logint(rng, 1, 100)
    types = rng.choice(["int8:1", "int4:1", "int2:1", "fp8:1", "fp16:1", "bf16:1", "fp32:1",
                        "fp16:1,int8:3,int4:4,int2:2", "int8:1,fp8:1,bf16:1,fp32:1"])
    dims = rng.choice(["128", "64", "32,64,128,256", "256,512", "ragged:4:1024", "ragged:4:64"])
    bags = rng.choice([f"fixed:{mean}", f"poisson:{mean}:1:128", f"uniform:{min(1, mean - 1)}:{2 * mean}"])
    if kind == "nobag":  # one width for every table
        dims = str(_logint(rng, 1, 32) * 16)
    layout = rng.randrange(1000)
    rows = _logint(rng, 1_000, 2_000_000)
    case = dict(kind=kind, tables=tables, rows_lo=max(16, rows // 4), rows_hi=rows, dims=dims, types=types,
                layout=layout, batch=batch, bags=bags, zipf=rng.choice([0.0, 1.05, 1.2]), tail=0.0,
                index=rng.choice(["int32", "int64"]),
                mode="none" if kind == "nobag" else rng.choice(["sum", "mean"]),
                out=rng.choice(["fp32", "fp16", "bf16"]),
                weighted=kind == "pooled" and rng.random() < 0.4)
    while True:  # no larger than the largest listed case, and a few GB of tables
        specs = _tables(case)
        n = case["batch"] * mean
        row_bytes = sum(_row_bytes(ty, d) for _, d, ty in specs)
        out_bytes = (n if kind == "nobag" else case["batch"]) * sum(4 * d for _, d, _ in specs)
        if n * row_bytes + out_bytes > 1.2e9 and case["batch"] > 1:
            case["batch"] //= 2
        elif sum(e * (_row_bytes(ty, d) + 16) for e, d, ty in specs) > 4e9:
            case["rows_lo"], case["rows_hi"] = max(16, case["rows_lo"] // 2), case["rows_hi"] // 2
        else:
            return case


# ------------------------------------------------------------------ sizes of a case

def _row_bytes(ty, dim):
    return dim * BITS[ty] // 8 + (4 if ty in INT_ROWS else 0)


def _tables(case):
    """[(rows, dim, type)] of the case: fixed by its own values."""
    rs = random.Random(case["layout"])
    kinds = [t.split(":") if ":" in t else (t, "1") for t in case["types"].split(",")]
    out = []
    for i in range(case["tables"]):
        rows = _logint(rs, case["rows_lo"], case["rows_hi"])
        ty = rs.choices([k for k, _ in kinds], [float(w) for _, w in kinds])[0]
        if case["dims"].startswith("ragged"):
            _, lo, hi = case["dims"].split(":")
            dim = _logint(rs, int(lo), int(hi))
        else:
            dim = int(rs.choice(case["dims"].split(",")))
        step = 32 // BITS[ty]  # a row fills whole 4-byte words
        out.append((rows, (dim + step - 1) // step * step, ty))
    return out


def _mean_len(rule):
    kind, *a = rule.split(":")
    return (float(a[0]) + float(a[1])) / 2 if kind == "uniform" else float(a[0])


def _feature_dims(case):
    rs = random.Random(case["layout"])
    dims = [int(rs.choice(case["dims"].split(","))) for _ in range(case["features"])]
    order = list(range(case["features"]))
    rs.shuffle(order)
    return dims, order


def _distinct_rows(rows, count, alpha):
    """Expected distinct rows among `count` draws from a table."""
    if alpha <= 0:
        return rows * -math.expm1(count * math.log1p(-1.0 / rows)) if rows > 1 else 1.0
    edges = np.unique(np.round(np.geomspace(1, rows + 1, 400)))
    mid, width = (edges[:-1] + edges[1:] - 1) / 2, np.diff(edges)
    p = mid ** -alpha
    p /= (p * width).sum()
    return float((width * -np.expm1(-count * p)).sum())


def work(case):
    """Bytes and operations one pass cannot do without: every distinct row touched, the other
    inputs once, the outputs once; a multiply and an add per element of every looked-up row."""
    if case["kind"] == "permute":
        return {"bytes": 4 * sum(_feature_dims(case)[0]) * case["batch"] * BITS[case["out"]] // 8, "flops": 0}
    isz = 8 if case["index"] == "int64" else 4
    if case["kind"] == "bucketize":
        rows = case["features"] * case["batch"]
        n = rows * _mean_len(case["lengths"])
        per = 2 * isz + (8 if case["weighted"] else 0) + (isz if case["sequence"] else 0) + \
            (isz if case["bucket_pos"] else 0)
        return {"bytes": int(n * per + rows * isz * (1 + case["ranks"])), "flops": 0}
    n = case["batch"] * _mean_len(case["bags"])
    nbytes = flops = 0.0
    for rows, dim, ty in _tables(case):
        per_out = n if case["kind"] == "nobag" else case["batch"]
        nbytes += _distinct_rows(rows, n, case["zipf"]) * _row_bytes(ty, dim)
        nbytes += n * (isz + (4 if case["weighted"] else 0)) + case["batch"] * isz
        nbytes += per_out * dim * BITS[case["out"]] // 8
        flops += 2 * n * dim
    return {"bytes": int(nbytes), "flops": int(flops)}


# ------------------------------------------------------------------ inputs

def _gen(seed, part=0):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1_000_003 + part * 7919 + 17) & 0x7FFF_FFFF_FFFF)
    return g


def _lengths(rule, n, g):
    """n lengths by the rule: the same set for every seed (so outputs keep their shape), in the seed's order."""
    kind, *a = rule.split(":")
    own = _gen(n, 1)
    if kind == "fixed":
        return torch.full((n,), int(a[0]), dtype=torch.int64, device="cuda")
    if kind == "uniform":
        lengths = torch.randint(int(a[0]), int(a[1]) + 1, (n,), device="cuda", generator=own)
        lengths[0].clamp_(min=1)  # at least one index in the call
    else:
        mean = torch.full((n,), float(a[0]), device="cuda")
        lengths = torch.poisson(mean, generator=own).to(torch.int64).clamp_(int(a[1]), int(a[2]))
    return lengths[torch.randperm(n, device="cuda", generator=g)]


def _ids(rows, count, alpha, tail, g):
    """Row ids: Zipf(alpha) ranks (inverse of the continuous CDF) scattered over the table, or uniform."""
    if alpha <= 0:
        return torch.randint(0, rows, (count,), device="cuda", generator=g)
    u = torch.rand(count, dtype=torch.float64, device="cuda", generator=g)
    e = 1.0 - alpha
    rank = ((((rows + 1.0) ** e - 1.0) * u + 1.0) ** (1.0 / e) - 1.0).to(torch.int64).clamp_(0, rows - 1)
    step = next(p for p in (1_000_003, 999_983, 7_368_787) if math.gcd(p, rows) == 1)
    ids = rank * step % rows
    if tail > 0:
        pick = torch.rand(count, device="cuda", generator=g) < tail
        ids = torch.where(pick, torch.randint(0, rows, (count,), device="cuda", generator=g), ids)
    return ids


def _payload(rows, dim, ty, g):
    """(payload bytes [rows, dim * bits / 8], fp16 (scale, bias) [rows, 2] or None) of one table."""
    if ty in INT_ROWS:
        # rows quantised between their min and max: bias about minus half the range
        codes = torch.randint(0, 256, (rows, dim * BITS[ty] // 8), dtype=torch.uint8, device="cuda", generator=g)
        span = torch.rand((rows, 2), device="cuda", generator=g) * 0.4 + 0.8
        scale = (span[:, 0] * 0.5 / (2 ** BITS[ty] - 1)).to(torch.float16)
        bias = (-0.25 * span[:, 1]).to(torch.float16)
        return codes, torch.stack([scale, bias], 1)
    vals = torch.randn((rows, dim), device="cuda", generator=g) * 0.1
    if ty == "fp8":  # 4 exponent bits, bias 7: below 2 the format is float8_e4m3
        return vals.to(torch.float8_e4m3fn).view(torch.uint8), None
    return vals.to(TORCH[ty]).view(torch.uint8), None


def _values(payload, header, dim, ty):
    """The table's values in 64 bits."""
    if ty not in INT_ROWS:
        dt = torch.float8_e4m3fn if ty == "fp8" else TORCH[ty]
        return payload.contiguous().view(dt).float().double()
    per = 8 // BITS[ty]
    shifts = torch.arange(per, device="cuda", dtype=torch.uint8) * BITS[ty]
    q = (payload[:, :, None] >> shifts) & (2 ** BITS[ty] - 1)
    h = header.double()
    return q.reshape(payload.shape[0], dim).double() * h[:, :1] + h[:, 1:]


def _sparse_inputs(case, seed):
    """indices, offsets, per-sample weights (or None), lengths [tables * batch] (int64)."""
    g = _gen(seed)
    n = case["tables"] * case["batch"]
    lengths = _lengths(case["bags"], n, g)
    per_table = lengths.view(case["tables"], -1).sum(1).cpu().tolist()
    ids = [_ids(rows, c, case["zipf"], case["tail"], g) for (rows, _, _), c in zip(_tables(case), per_table)]
    dt = TORCH[case["index"]]
    offsets = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=offsets[1:])
    ids = torch.cat(ids).to(dt)
    psw = torch.rand(ids.numel(), device="cuda", generator=g) if case["weighted"] else None
    return ids, offsets.to(dt), psw, lengths


def _prepare_tbe(case, seed):
    pkg = load_package()
    st = {t.name.lower(): t for t in pkg.SparseType}
    specs = _tables(case)
    mode = pkg.PoolingMode[case["mode"].upper()]
    module = pkg.IntNBitTableBatchedEmbeddingBagsCodegen(
        [(rows, dim, st[ty]) for rows, dim, ty in specs], device="cuda", pooling_mode=mode,
        output_dtype=st[case["out"]], indices_dtype=TORCH[case["index"]])
    for t, ((rows, dim, ty), (payload, header)) in enumerate(zip(specs, module.split_embedding_weights())):
        codes, sb = _payload(rows, dim, ty, _gen(seed, 1 + t))
        payload.copy_(codes)
        if sb is not None:
            header.copy_(sb.view(torch.uint8))
    indices, offsets, psw, _ = _sparse_inputs(case, seed)
    return {"kind": "tbe", "module": module, "indices": indices, "offsets": offsets, "psw": psw}


def _exact_tbe(case, seed):
    indices, _, psw, lengths = _sparse_inputs(case, seed)
    specs, B = _tables(case), case["batch"]
    per_table = lengths.view(len(specs), B)
    outs, first = [], 0
    for t, (rows, dim, ty) in enumerate(specs):
        vals = _payload(rows, dim, ty, _gen(seed, 1 + t))
        n = int(per_table[t].sum())
        idx = indices[first:first + n].long()
        used, where = torch.unique(idx, return_inverse=True)
        x = _values(vals[0][used], None if vals[1] is None else vals[1][used], dim, ty)
        if case["kind"] == "nobag":
            outs.append(x[where])
        else:
            acc = torch.zeros((B, dim), dtype=torch.float64, device="cuda")
            bag = torch.repeat_interleave(torch.arange(B, device="cuda"), per_table[t])
            for a in range(0, n, 1 << 19):
                part = x[where[a:a + (1 << 19)]]
                if psw is not None:
                    part = part * psw[first + a:first + a + part.shape[0], None].double()
                acc.index_add_(0, bag[a:a + (1 << 19)], part)
            if case["mode"] == "mean":
                acc /= per_table[t].clamp(min=1)[:, None]
            outs.append(acc)
        first += n
    return [torch.cat(outs, 0 if case["kind"] == "nobag" else 1)]


def _permute_inputs(case, seed):
    dims, order = _feature_dims(case)
    g = _gen(seed)
    x, grad = (torch.randn((case["batch"], sum(dims)), device="cuda", generator=g).to(TORCH[case["out"]])
               for _ in range(2))
    return dims, order, x, grad


def _prepare_permute(case, seed):
    dims, order, x, grad = _permute_inputs(case, seed)
    perm = load_package().PermutePooledEmbeddings(dims, order, device=torch.device("cuda"))
    return {"kind": "permute", "perm": perm, "x": x.requires_grad_(), "grad": grad}


def _exact_permute(case, seed):
    dims, order, x, grad = _permute_inputs(case, seed)
    starts = np.concatenate([[0], np.cumsum(dims)])
    cols = torch.from_numpy(np.concatenate([np.arange(starts[f], starts[f + 1]) for f in order])).cuda()
    back = torch.empty_like(grad)
    back[:, cols] = grad
    return [x[:, cols].double(), back.double()]


def _bucketize_inputs(case, seed):
    g = _gen(seed)
    F, B, R = case["features"], case["batch"], case["ranks"]
    dt = TORCH[case["index"]]
    lengths = _lengths(case["lengths"], F * B, g)
    lo, hi = map(int, case["blocks"].split(":"))
    blocks = torch.randint(lo, hi + 1, (F,), device="cuda", generator=g)
    pos = None
    if case["positions"]:  # uneven shards of the same feature: boundaries 0 = p0 < p1 < ... < pR
        steps = torch.randint(1, hi + 1, (F, R), device="cuda", generator=g)
        pos = torch.cat([torch.zeros((F, 1), dtype=torch.int64, device="cuda"), steps.cumsum(1)], 1)
    limit = blocks * R if pos is None else pos[:, -1]
    per = lengths.view(F, B).sum(1)
    u = torch.rand(int(per.sum()), dtype=torch.float64, device="cuda", generator=g)
    span = torch.repeat_interleave(limit, per)
    indices = (u * span).to(torch.int64).clamp_(max=span - 1)
    w = torch.rand(indices.numel(), device="cuda", generator=g) if case["weighted"] else None
    return lengths.to(dt), indices.to(dt), blocks.to(dt), w, pos


def _prepare_bucketize(case, seed):
    load_package()
    lengths, indices, blocks, w, pos = _bucketize_inputs(case, seed)
    lists = None if pos is None else [p.to(indices.dtype).contiguous() for p in pos]
    return {"kind": "bucketize", "case": case, "args": (lengths, indices, case["bucket_pos"], case["sequence"],
                                                        blocks, case["ranks"], w, None, -1, lists)}


def _exact_bucketize(case, seed):
    lengths, indices, blocks, w, pos = _bucketize_inputs(case, seed)
    F, B, R = case["features"], case["batch"], case["ranks"]
    L = F * B
    row = torch.repeat_interleave(torch.arange(L, device="cuda"), lengths.long())
    idx, f = indices.long(), row // B
    if pos is None:
        bucket = idx // blocks.long()[f]
        local = idx - bucket * blocks.long()[f]
    else:
        bucket = torch.zeros_like(idx)
        for r in range(1, R):
            bucket += idx >= pos[f, r]
        local = idx - pos[f, bucket]
    seg = bucket * L + row
    order = torch.sort(seg, stable=True).indices
    out = [torch.bincount(seg, minlength=R * L), local[order]]
    if w is not None:
        out.append(w[order].double())
    if case["bucket_pos"]:
        start = torch.cumsum(lengths.long(), 0) - lengths.long()
        out.append((torch.arange(idx.numel(), device="cuda") - start[row])[order])
    if case["sequence"]:
        unb = torch.empty_like(order)
        unb[order] = torch.arange(order.numel(), device="cuda")
        out.append(unb)
    return out


# ------------------------------------------------------------------ the interface

def prepare(case, seed):
    """What the user's program holds before the call: inputs, and the module it keeps."""
    if case["kind"] == "permute":
        return _prepare_permute(case, seed)
    if case["kind"] == "bucketize":
        return _prepare_bucketize(case, seed)
    return _prepare_tbe(case, seed)


def run(state):
    """One pass; the outputs as a list."""
    if state["kind"] == "tbe":
        return [state["module"](state["indices"], state["offsets"], state["psw"])]
    if state["kind"] == "permute":
        out = state["perm"](state["x"])
        (dx,) = torch.autograd.grad(out, state["x"], state["grad"])
        return [out.detach(), dx]
    return [t for t in torch.ops.fbgemm.block_bucketize_sparse_features(*state["args"]) if t is not None]


def tolerance(case):
    """Copies and whole numbers are exact.  Sums in 32 bits differ by their order; 16-bit results
    differ where the rounding of that sum falls on the other side (about four times what two
    orders, or the 64-bit sum, were measured to differ)."""
    if case["kind"] in ("permute", "bucketize"):
        return "exact"
    return {"rel": {"fp32": 2e-6, "fp16": 1e-3, "bf16": 8e-3}[case["out"]]}


def exact(case, seed):
    """What run() returns, in 64 bits by plain torch."""
    if case["kind"] == "permute":
        return _exact_permute(case, seed)
    if case["kind"] == "bucketize":
        return _exact_bucketize(case, seed)
    return _exact_tbe(case, seed)
