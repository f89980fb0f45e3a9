"""The work that users of engine_amd have it do, as cases to be timed.

Every case goes through the package's public calls on device-resident
columns: fused select + sum (one column, one batch of columns), the codecs
in both directions, and chains of operators (eager and as a recorded plan).
Formats, value distributions and sizes are those of bench.py, datagen.py
and the tests; the values are drawn on the GPU.

A column's image is returned as the device words that the format defines:
the compressed part and the raw rest (the gap between them is undefined),
with its meta data, which the caller reads to know their sizes.
"""
import ctypes
import math

import torch

import engine_amd as ea
from engine_amd import hip
from engine_amd.formats import (BatchConfig, MS_CMP_EQ, MS_CMP_GE, MS_CMP_LT, MS_RLE, MS_UNCOMPR,
                                default_delta_dynamic_vbp_f, default_for_dynamic_vbp_f, dynamic_vbp_f, rle_f,
                                static_vbp_f, uncompr_f)

DEV = "cuda:0"
CMP = {"eq": MS_CMP_EQ, "lt": MS_CMP_LT, "ge": MS_CMP_GE}
KINDS = ("static_vbp", "dynamic_vbp", "delta", "for", "rle")
# compressed bytes per value of each kind's distribution below
BYTES = {"static_vbp": 2.0, "dynamic_vbp": 2.0625, "delta": 1.0625, "for": 2.07, "rle": 0.25}
# the work-queue shape that bench.py's sweep runs at
SWEEP_SHAPE = dict(wg_per_cu=4, units_per_item=32, tiles_per_item=8, runs_per_item=4096, values_per_item=2048)


def listed():
    return [
        # one selective sum over a short column: the latency of a fused call
        {"name": "sum_small", "op": "sum", "kind": "dynamic_vbp", "n": 1000, "cmp": "lt"},
        # the format cascade: four long columns of four formats, one batch
        {"name": "batch_sweep", "op": "batch_sweep", "n": 1 << 27},
        # a table's many uneven columns of five formats, one batch
        {"name": "batch_uneven", "op": "batch_uneven", "cols": 1024, "lo": 1000, "hi": 1000000},
        # a short column stored and read back: latency of the codecs
        {"name": "roundtrip_small", "op": "roundtrip", "kind": "delta", "n": 10007},
        # loading columns: an ordinary one, a long ragged one, a column of runs
        {"name": "compress_dvbp", "op": "compress", "kind": "dynamic_vbp", "n": 1 << 24},
        {"name": "compress_for", "op": "compress", "kind": "for", "n": 100000077},
        {"name": "compress_rle", "op": "compress", "kind": "rle", "n": 1 << 26},
        # reading columns back: sorted keys, and runs of a ragged column
        {"name": "decompress_delta", "op": "decompress", "kind": "delta", "n": 1 << 27},
        {"name": "decompress_rle", "op": "decompress", "kind": "rle", "n": 50000003},
        # the reference's benchmark query, its operators one by one
        {"name": "query_static", "op": "query", "n": 1 << 24, "bw": 12, "step": 1},
        # the two-column query as a recorded plan
        {"name": "plan_query", "op": "plan", "rows": 1 << 28},
        # the OR of two predicates' position lists, its rows fetched and summed
        {"name": "union_fetch", "op": "union", "rows": (1 << 25) + 4093},
    ]


def _log_int(rng, lo, hi):
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    # odd sizes, whole blocks and whole pages all occur
    unit = rng.choice((1, 1, 1, 512, 2048))
    return max(lo, n // unit * unit) if n >= 4 * unit else n


def draw(rng):
    op = rng.choice(("sum", "sum", "batch_sweep", "batch_uneven", "roundtrip", "compress", "compress", "decompress",
                     "decompress", "query", "plan", "union"))
    if op == "sum":
        return {"op": op, "kind": rng.choice(KINDS), "n": _log_int(rng, 1000, 1 << 27), "cmp": rng.choice(tuple(CMP))}
    if op == "batch_sweep":
        return {"op": op, "n": _log_int(rng, 1 << 20, 1 << 27)}
    if op == "batch_uneven":
        return {"op": op, "cols": _log_int(rng, 64, 1024), "lo": 1000, "hi": rng.choice((100000, 300000, 1000000))}
    if op == "roundtrip":
        return {"op": op, "kind": rng.choice(KINDS), "n": _log_int(rng, 1000, 200000)}
    if op == "compress":
        return {"op": op, "kind": rng.choice(KINDS), "n": _log_int(rng, 100000, 1 << 27)}
    if op == "decompress":
        return {"op": op, "kind": rng.choice(KINDS), "n": _log_int(rng, 100000, 1 << 27)}
    if op == "query":
        return {"op": op, "n": _log_int(rng, 1 << 18, 1 << 25), "bw": rng.randint(4, 24), "step": rng.choice((1, 8))}
    if op == "plan":
        return {"op": op, "rows": _log_int(rng, 1 << 20, 1 << 28)}
    return {"op": op, "rows": _log_int(rng, 1 << 18, 1 << 26)}


# ---------------------------------------------------------------- values
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _bits(g, n, bits):
    """n values uniform in [0, 2^bits)."""
    return torch.randint(0, 1 << bits, (n,), generator=g, device=DEV, dtype=torch.int64)


def _geometric(g, n, p):
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64).clamp_(min=1e-300)
    return (u.log_() / math.log1p(-p)).floor_().add_(1).to(torch.int64)


def _values(kind, g, n, bw=16):
    """(values, select value): the distribution that suits each format, as
    datagen's, and a value that about half of them are below.  The widths,
    gaps and runs are shuffled, not their numbers: a length has one
    compressed size."""
    if kind == "static_vbp":
        return _bits(g, n, bw), 1 << (bw - 1)
    if kind == "dynamic_vbp":
        # a bit width of its own per 512 values, the top bit set once
        nb = n // 512
        b = (torch.randperm(nb, generator=g, device=DEV) % 32 + 1).reshape(nb, 1)
        x = torch.randint(0, 1 << 32, (nb, 512), generator=g, device=DEV, dtype=torch.int64)
        x >>= 32 - b
        at = torch.randint(0, 512, (nb, 1), generator=g, device=DEV, dtype=torch.int64)
        x.scatter_(1, at, x.gather(1, at) | (torch.ones_like(b) << (b - 1)))
        x = x.reshape(-1)
        return (x if n % 512 == 0 else torch.cat([x, _bits(g, n % 512, 16)])), 1 << 16
    if kind == "delta":
        # sorted keys, gaps of at most 31 and eight of 16 in a row per 512
        x = _geometric(g, n, 0.1).clamp_(max=31)
        at = torch.arange(0, n // 512 * 512, 512, device=DEV).reshape(-1, 1) + torch.arange(256, 264, device=DEV)
        x[at.reshape(-1)] = 16
        x[0] = 0
        x = torch.cumsum(x, 0)
        return x, int(x[n // 2])
    if kind == "for":
        base = (1 << 40) + int(torch.randint(0, 1 << 40, (1,), generator=g, device=DEV))
        x = _bits(g, n, 16)
        # both ends of the offsets' range occur in every 1024 values
        ends = torch.arange(0, n // 1024 * 1024, 1024, device=DEV)
        x[ends + 77], x[ends + 400], x[ends + 900] = 0, 65535, 65535
        return x + base, base + (1 << 15)
    # n / 64 runs between random cuts, neighbours of different values
    runs = max(1, n // 64)
    cuts = torch.rand(n, generator=g, device=DEV)
    cuts[0] = -1
    starts = torch.zeros(n, dtype=torch.int64, device=DEV)
    starts[torch.topk(cuts, runs, largest=False).indices if runs < 1024 else torch.sort(cuts).indices[:runs]] = 1
    ids = torch.cumsum(starts, 0) - 1
    vals = 2 * _bits(g, runs, 19) + (torch.arange(runs, device=DEV) & 1)
    return vals[ids], 1 << 19


def _format(kind, bw=16):
    return {"static_vbp": static_vbp_f(bw, 8), "dynamic_vbp": dynamic_vbp_f(512, 2048, 8),
            "delta": default_delta_dynamic_vbp_f(8), "for": default_for_dynamic_vbp_f(8), "rle": rle_f()}[kind]


def _flags(g, n):
    """Zipf(1.1) over 8 values."""
    w = torch.tensor([1.0 / (k + 1) ** 1.1 for k in range(8)], dtype=torch.float64)
    cdf = torch.cumsum(w / w.sum(), 0).to(device=DEV, dtype=torch.float32)
    return torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV), right=True).clamp_(max=7)


def _union_inputs(case, g):
    """(flag, key, measure, rows of either predicate): 9% of the rows have
    flag 3, 25% a key below 2^18, 2% both, in random places."""
    n = case["rows"]
    r = torch.randperm(n, generator=g, device=DEV)
    a0, b0, b1 = 9 * n // 100, 7 * n // 100, 32 * n // 100
    flag = _flags(g, n)
    flag = torch.where(r < a0, 3, torch.where(flag == 3, 2, flag))
    key = _bits(g, n, 20)
    key = torch.where((r >= b0) & (r < b1), key % (1 << 18), key | (1 << 18))
    return flag, key, _bits(g, n, 16), b1


# ---------------------------------------------------------------- columns
def _column(x, fmt=None):
    raw = ea.from_device(x.data_ptr(), x.numel())
    return raw if fmt is None else ea.morph(fmt, raw)


class _Words:
    """`n` device words at `ptr`, for torch; keeps their owner alive."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i8", "data": (ptr, False), "version": 3,
                                         "strides": None}


def _words(owner, ptr, n):
    if n == 0:
        return torch.empty(0, dtype=torch.int64, device=DEV)
    return torch.as_tensor(_Words(owner, ptr, n), device=DEV)


def _raw_words(col, n):
    """The n values of an uncompr_f column whose count the caller knows."""
    return _words(col, col.device_ptr, n)


def _gap(fmt):
    """The gap in front of an image's raw rest: two blocks' largest size."""
    if fmt.kind in (MS_UNCOMPR, MS_RLE):
        return 0
    out = ctypes.c_uint64()
    ea.check(ea.lib().ms_size_max_byte(ctypes.byref(fmt), fmt.block_size(), ctypes.byref(out)))
    return 2 * out.value


def _image(col, gap, stream=None):
    """A column's whole image and its meta data."""
    m = col.meta(stream)
    p = col.device_ptr
    out = {"meta": [m.count, m.size_used, m.size_compr], "main": _words(col, p, m.size_compr // 8)}
    if m.size_used != m.size_compr:
        at = (m.size_compr + gap + 63) // 64 * 64
        out["rest"] = _words(col, p + at, (m.size_used - at) // 8)
    return out


# ---------------------------------------------------------------- cases
def _uneven(case, g):
    """(kind, bit width, length) of every column."""
    n = case["cols"]
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    lens = (lo + u * (hi - lo)).exp().to(torch.int64).tolist()
    kinds = torch.randint(0, 5, (n,), generator=g, device=DEV).tolist()
    bws = torch.randint(1, 33, (n,), generator=g, device=DEV).tolist()
    return [(KINDS[k], b, m) for k, b, m in zip(kinds, bws, lens)]


def _batch_inputs(case, g):
    """Yields (format, values, select value) of every column of a batch."""
    if case["op"] == "batch_sweep":
        for kind in ("dynamic_vbp", "delta", "for", "rle"):
            x, val = _values(kind, g, case["n"])
            yield _format(kind), x, val
    else:
        for kind, bw, n in _uneven(case, g):
            x, val = _values(kind, g, n, bw)
            yield _format(kind, bw), x, val


def _plan_inputs(case, g):
    n = case["rows"]
    return _flags(g, n), _bits(g, n, 20), _bits(g, n, 16)


def prepare(case, seed):
    ea.init(0)
    g, op = _gen(seed), case["op"]
    st = {"op": op}
    if op == "sum":
        x, val = _values(case["kind"], g, case["n"])
        st["col"], st["cmp"] = _column(x, _format(case["kind"])), CMP[case["cmp"]]
        st["val"] = int(x[case["n"] // 3]) if case["cmp"] == "eq" else val
        st["res"] = ea.DeviceU64()
        st["out"] = _words(st["res"], st["res"].p.value, 1)
    elif op in ("batch_sweep", "batch_uneven"):
        b = ea.Batch()
        for fmt, x, val in _batch_inputs(case, g):
            b.enqueue(_column(x, fmt), CMP["lt"], val)
        if op == "batch_sweep":
            b.config = BatchConfig(**SWEEP_SHAPE)
        res = ea.DeviceU64(len(b))
        b.run(res)      # builds the work queue
        st["batch"], st["res"], st["out"] = b, res, _words(res, res.p.value, len(b))
    elif op in ("roundtrip", "compress", "decompress"):
        fmt = _format(case["kind"])
        x, _ = _values(case["kind"], g, case["n"])
        st["fmt"], st["gap"], st["n"] = fmt, _gap(fmt), case["n"]
        st["col"] = _column(x, fmt if op == "decompress" else None)
    elif op == "query":
        fmt = static_vbp_f(case["bw"], case["step"])
        st["col"] = _column(_bits(g, case["n"], case["bw"]), fmt)
        st["lanes"], st["val"] = case["step"], 1 << (case["bw"] - 1)
    elif op == "plan":
        cols = [_column(x, dynamic_vbp_f(512, 2048, 8)) for x in _plan_inputs(case, g)]
        hip.synchronize()
        stream, plan = hip.Stream(), ea.Plan()
        for _ in range(2):       # measure, then capture
            with plan.record(stream):
                res, lists = _plan_query(cols, stream)
        # the plan's columns live in its arena: its owner outlives the result
        st.update(plan=plan, stream=stream, out=_words((plan, cols, lists, res), res.device_ptr, 1))
    else:
        f, key, ms, st["count"] = _union_inputs(case, g)
        lfmt = default_delta_dynamic_vbp_f(8)
        st["l"] = ea.select(MS_CMP_EQ, 3, lfmt, _column(f, dynamic_vbp_f(512, 2048, 8)))
        st["r"] = ea.select(MS_CMP_LT, 1 << 18, lfmt, _column(key, dynamic_vbp_f(512, 2048, 8)))
        st["col"], st["fmt"] = _column(ms, dynamic_vbp_f(512, 2048, 8)), lfmt
    return st


def _plan_query(cols, stream):
    """select(flag == 3) and select(key < 2^18) -> intersect -> project
    (measure) -> agg_sum."""
    f = default_delta_dynamic_vbp_f(8)
    p1 = ea.select(MS_CMP_EQ, 3, f, cols[0], 8, stream)
    p2 = ea.select(MS_CMP_LT, 1 << 18, f, cols[1], 8, stream)
    both = ea.intersect_sorted(f, p1, p2, stream)
    m = ea.project(uncompr_f(), cols[2], both, 8, stream)
    return ea.agg_sum(m, stream), (p1, p2, both, m)


def run(st):
    op = st["op"]
    if op == "sum":
        ea.select_sum(st["cmp"], st["val"], st["col"], st["res"])
        return st["out"]
    if op in ("batch_sweep", "batch_uneven"):
        st["batch"].run(st["res"])
        return st["out"]
    if op == "compress":
        return _image(ea.morph(st["fmt"], st["col"]), st["gap"])
    if op == "decompress":
        return _raw_words(ea.morph(uncompr_f(), st["col"]), st["n"])
    if op == "roundtrip":
        c = ea.morph(st["fmt"], st["col"])
        return {"image": _image(c, st["gap"]), "values": _raw_words(ea.morph(uncompr_f(), c), st["n"])}
    if op == "query":
        pos = ea.select(MS_CMP_LT, st["val"], uncompr_f(), st["col"], st["lanes"])
        dat = ea.project(uncompr_f(), st["col"], pos, st["lanes"])
        return _raw_words(ea.agg_sum(dat), 1)
    if op == "plan":
        st["plan"].launch(st["stream"])
        return st["out"]
    both = ea.merge_sorted(st["fmt"], st["l"], st["r"])
    dat = ea.project(uncompr_f(), st["col"], both)
    return {"sum": _raw_words(ea.agg_sum(dat), 1), "values": _raw_words(dat, st["count"])}


def work(case):
    op, ops = case["op"], 0
    if op == "sum":
        b = case["n"] * BYTES[case["kind"]] + 8
        ops = case["n"] * 2
    elif op == "batch_sweep":
        b = case["n"] * sum(BYTES[k] for k in ("dynamic_vbp", "delta", "for", "rle")) + 32
        ops = case["n"] * 8
    elif op == "batch_uneven":
        values = case["cols"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        b = values * sum(BYTES.values()) / 5 + 8 * case["cols"]
        ops = values * 2
    elif op in ("compress", "decompress"):
        b = case["n"] * (8 + BYTES[case["kind"]])
    elif op == "roundtrip":
        b = case["n"] * (16 + 2 * BYTES[case["kind"]])
    elif op == "query":
        # the column, the positions written and read, the fetched codes, the
        # fetched values written and read
        b = case["n"] * (case["bw"] / 8 * 1.5 + 0.5 * 8 * 4)
        ops = case["n"] * 1.5
    elif op == "plan":
        # flags (3 bits), keys (20), the lists (9% and 25% of the rows, 9
        # bits a position) and their common rows, the fetched measures
        b = case["rows"] * (3 / 8 + 20 / 8 + 2 * (0.087 + 0.25 + 0.022) * 9 / 8 + 0.022 * 18)
        ops = case["rows"] * 4
    else:
        b = case["rows"] * ((0.087 + 0.25 + 2 * 0.315) * 9 / 8 + 0.315 * (2 + 16))
        ops = case["rows"]
    return {"bytes": float(b), "flops": float(ops)}


def _sum_of(x, cmp, val):
    m = x == val if cmp == "eq" else x < val if cmp == "lt" else x >= val
    return torch.where(m, x, 0).sum().reshape(1)


def exact(case, seed):
    g, op = _gen(seed), case["op"]
    if op == "sum":
        x, val = _values(case["kind"], g, case["n"])
        return _sum_of(x, case["cmp"], int(x[case["n"] // 3]) if case["cmp"] == "eq" else val)
    if op in ("batch_sweep", "batch_uneven"):
        return torch.cat([_sum_of(x, "lt", val) for _, x, val in _batch_inputs(case, g)])
    if op == "decompress":
        return _values(case["kind"], g, case["n"])[0]
    if op == "query":
        return _sum_of(_bits(g, case["n"], case["bw"]), "lt", 1 << (case["bw"] - 1))
    if op == "plan":
        f, key, ms = _plan_inputs(case, g)
        return torch.where((f == 3) & (key < (1 << 18)), ms, 0).sum().reshape(1)
    if op == "union":
        f, key, ms, _ = _union_inputs(case, g)
        v = ms[(f == 3) | (key < (1 << 18))]
        return {"sum": v.sum().reshape(1), "values": v}
    return None      # images: bytes of the format, no numbers
