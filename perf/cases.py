"""Performance cases of the library, each one pass through its public entry points.

A case is a dict: "kind" says which part of the library it runs, the rest its
sizes and options.  Kinds:

  q11     fused decode + filter + SUM (Q1.1 shape) over an encoded fact table
  star    fused decode + joins + group-by (Q2.1, Q3.1, Q4.1 shapes)
  unpack  a fixed-width column to plain values, with or without the checksum
  decode  a column of any encoding to plain values, in row or stored order
  encode  plain values to a column: a fixed scheme, or one chosen per vector
  batch   many uneven segments range-counted in one launch
  train   one training step of the selector's network (gradient and Adam)

The tables are the synthetic ones the benchmark uses (fls.gen_*), or columns
of the same kinds made with torch from the seed.
"""
import math

import numpy as np
import torch

import fastlanesgpu_amd as fls
from fastlanesgpu_amd import selector

VECTOR = fls.VECTOR_SIZE


def listed():
    return [
        # the headline scan: SSB Q1.1 over a resident fact table
        {"name": "q11_120m", "kind": "q11", "rows": 120_000_000, "columns": "ssb", "pred_load": False},
        # the same query over one small chunk: what a call costs by itself
        {"name": "q11_100k", "kind": "q11", "rows": 100_003, "columns": "ssb", "pred_load": False},
        # Q1.1 over columns whose vectors each carry their own encoding, as the
        # per-vector encoders write them, at the row count of SSB SF10
        {"name": "q11_mixed_sf10", "kind": "q11", "rows": 59_986_214, "columns": "mixed", "pred_load": False},
        # the selective star join: two semi-joins, few survivors
        {"name": "q21_120m", "kind": "star", "query": "q21", "rows": 120_000_000, "columns": "ssb"},
        # the widest star join: six fact columns, four dimensions, SF10
        {"name": "q41_sf10", "kind": "star", "query": "q41", "rows": 59_986_214, "columns": "ssb"},
        # plain bit-unpack with its checksum at the benchmark's size
        {"name": "unpack_bw11_16m", "kind": "unpack", "bw": 11, "values": 1 << 24, "checksum": True},
        # a sorted key column handed to an operator downstream in row order
        {"name": "decode_delta_120m", "kind": "decode", "scheme": "delta", "data": "orderkeys", "rows": 120_000_000,
         "order": "rows", "via": "column"},
        # a run-length column (mean run 8) in row order, ragged end
        {"name": "decode_rle_67m", "kind": "decode", "scheme": "rle", "data": "runs", "rows": (1 << 26) + 777,
         "order": "rows", "via": "column"},
        # loading a sorted column: plan, allocation of the words, pack
        {"name": "encode_delta_sf10", "kind": "encode", "scheme": "delta", "data": "orderkeys", "rows": 59_986_214},
        # loading a measure column with the trained selector
        {"name": "encode_learned_120m", "kind": "encode", "scheme": "learned", "data": "prices",
         "rows": 120_000_000},
        # a file's worth of column chunks of every encoding and width
        {"name": "batch_4096", "kind": "batch", "segments": 4096, "log2_min": 10, "log2_max": 24,
         "tile_vectors": 128, "dynamic": True},
        # one step of the selector's training at the benchmark's batch
        {"name": "train_4096", "kind": "train", "samples": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["q11", "star", "unpack", "decode", "decode", "encode", "encode", "batch", "train"])
    rows = _log_int(rng, 2_000, 120_000_000)
    if kind == "q11":
        return {"kind": kind, "rows": rows, "columns": rng.choice(["ssb", "ssb", "mixed"]),
                "pred_load": rng.random() < 0.25}
    if kind == "star":
        query = rng.choice(["q21", "q21_pht", "q31", "q41"])  # hash-table probes take bit-packed columns only
        columns = "ssb" if query == "q21_pht" else rng.choice(["ssb", "ssb", "ssb", "mixed"])
        return {"kind": kind, "query": query, "rows": rows, "columns": columns}
    if kind == "unpack":
        return {"kind": kind, "bw": rng.randint(1, 32), "values": rows, "checksum": rng.random() < 0.5}
    if kind == "decode":
        scheme = rng.choice(["bitpack", "delta", "rle", "mixed"])
        order = rng.choice(["rows", "stored"])
        via = rng.choice(["column", "direct"]) if order == "stored" and scheme != "bitpack" else "column"
        return {"kind": kind, "scheme": scheme, "data": rng.choice(DATA_OF[scheme]), "rows": rows, "order": order,
                "via": via}
    if kind == "encode":
        scheme = rng.choice(["bitpack", "delta", "rle", "exhaustive", "learned"])
        return {"kind": kind, "scheme": scheme, "data": rng.choice(DATA_OF[scheme]), "rows": rows}
    if kind == "batch":
        return {"kind": kind, "segments": _log_int(rng, 64, 2048), "log2_min": 10, "log2_max": rng.randint(16, 24),
                "tile_vectors": rng.choice([32, 64, 128, 256]), "dynamic": rng.random() < 0.7}
    return {"kind": kind, "samples": _log_int(rng, 256, 65_536)}


# ------------------------------------------------------------------- columns
# What each scheme meets: a user bit-packs measures, delta-codes sorted
# columns, run-length codes clustered ones, and leaves the choice per vector
# to the selector for anything.
DATA_OF = {
    "bitpack": ["quantities", "prices"],
    "delta": ["orderkeys", "timestamps"],
    "rle": ["runs", "orderkeys"],
    "mixed": ["families", "prices", "orderkeys", "runs"],
    "exhaustive": ["families", "prices", "orderkeys", "runs"],
    "learned": ["families", "prices", "orderkeys", "runs"],
}
BITS_OF = {"quantities": 6, "prices": 24}


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _random(n, top, g):
    return torch.randint(0, top, (n,), generator=g, device="cuda", dtype=torch.int32)


def _values(data, n, seed):
    """n uint32 values (int32 tensor) of a column as a table would hold it."""
    if data in ("quantities", "prices"):
        return fls.gen_c2(seed, n)[1 if data == "quantities" else 3]
    if data == "families":  # uniform, Zipf, noisy sorted and run vectors in turn
        nv = selector.n_vectors(n)
        return selector.gen_train_vectors(seed, 0, nv)[:n]
    g = _rng(seed)
    if data == "orderkeys":  # sorted, about four rows a key
        return torch.cumsum(_random(n, 4, g) == 0, 0, dtype=torch.int32) + 1
    if data == "timestamps":  # sorted, steps of 0..15
        return torch.cumsum(_random(n, 16, g), 0, dtype=torch.int32) + 1_000_000
    if data == "runs":  # clustered: runs of mean length 8, 16-bit values
        run = torch.cumsum(_random(n, 8, g) == 0, 0, dtype=torch.int32)
        return _random(n, 1 << 16, g)[run.long()]
    raise ValueError(data)


def _fixed(values, n, bw, base=0, transposed=False):
    words = fls.pack_column_device(values, n, bw, base=base, transposed=transposed)
    return fls.Column(fls.ENC_BITPACK, n, words, bw=bw, base=base, transposed=transposed,
                      n_words=fls.packed_words(n, bw))


def _delta(values, n):
    words, vmeta, bases = fls.delta_encode_device(values, n)
    return fls.Column(fls.ENC_DELTA, n, words, vmeta=vmeta, bases=bases)


def _rle(values, n):
    words, vmeta, rmeta, bases = fls.rle_encode_device(values, n)
    return fls.Column(fls.ENC_RLE, n, words, vmeta=vmeta, bases=bases, aux=rmeta)


def _mixed(values, n):
    ws = selector.MixedWorkspace(n)
    selector.mixed_encode_exhaustive(values, n, ws)
    c = ws.column(n)
    return fls.Column(fls.ENC_MIXED, n, c.words.clone(), vmeta=c.vmeta, aux=c.aux, n_words=c.n_words)


def _column(case, seed):
    n, data = case["rows"], case["data"]
    x = _values(data, n, seed)
    if case["scheme"] == "bitpack":
        return _fixed(x, n, BITS_OF[data], transposed=True)
    return {"delta": _delta, "rle": _rle, "mixed": _mixed}[case["scheme"]](x, n)


def _q11_table(n, columns, seed):
    od, qty, disc, price = fls.gen_c2(seed, n)
    if columns == "mixed":
        return [_mixed(c, n) for c in (od, qty, disc, price)]
    return [_delta(od, n)] + [_fixed(c, n, bw, transposed=True) for c, bw in ((qty, 6), (disc, 4), (price, 24))]


def _star_table(query, n, columns, seed):
    """The query's fact columns and dimensions (1-based keys, as in the benchmark's table)."""
    f = fls.gen_c3_fact(seed, n, with_customer=True)
    extra = fls.gen_star_extra(seed, n)
    dims = fls.gen_c3_dims(seed)
    dims["p_mfgr"] = extra["p_mfgr"]
    spec = {  # values, first value, width
        "date": (f["datefk"], 1, 12), "cust": (f["custfk"], 1, 20), "supp": (f["suppfk"], 1, 16),
        "part": (f["partfk"], 1, 20), "rev": (f["revenue"], 0, 24), "cost": (extra["supplycost"], 60_000, 16)}
    names = {"q31": ("date", "cust", "supp", "rev"), "q41": ("date", "cust", "supp", "part", "rev", "cost")}.get(
        query, ("date", "supp", "part", "rev"))
    cols = []
    for k in names:
        x, base, bw = spec[k]
        x = x + 1 if base == 1 else x
        cols.append(_mixed(x, n) if columns == "mixed" else _fixed(x, n, bw, base=base))
    return cols, dims


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "q11":
        s["cols"] = _q11_table(case["rows"], case["columns"], seed)
        s["out"] = torch.zeros(2, dtype=torch.int64, device="cuda")
    elif kind == "star":
        q = case["query"]
        s["cols"], s["dims"] = _star_table(q, case["rows"], case["columns"], seed)
        if q == "q21_pht":
            s["pht"], s["keep"] = fls.q21_build_pht(s["dims"])
        else:
            s["ws"] = {"q21": fls.q21_build, "q31": fls.q31_build, "q41": fls.q41_build}[q](s["dims"])
        slots = {"q31": 4375, "q41": 175}.get(q, 7000)
        s["out"] = torch.zeros(2 * slots, dtype=torch.int64, device="cuda")
    elif kind == "unpack":
        n, bw = case["values"], case["bw"]
        s["words"] = fls.pack_column_device(fls.gen_c1(seed, n, bw), n, bw)
        s["n_vec"] = selector.n_vectors(n)
        s["out"] = torch.empty(s["n_vec"] * VECTOR, dtype=torch.int32, device="cuda")
        s["checksum"] = fls.checksum_buffer()
    elif kind == "decode":
        s["col"] = _column(case, seed)
        s["n_vec"] = selector.n_vectors(case["rows"])
        s["out"] = torch.empty(s["n_vec"] * VECTOR, dtype=torch.int32, device="cuda")
    elif kind == "encode":
        s["x"] = _values(case["data"], case["rows"], seed)
        if case["scheme"] in ("exhaustive", "learned"):
            s["ws"] = selector.MixedWorkspace(case["rows"])
        if case["scheme"] == "learned":
            s["selector"] = selector.LearnedSelector.trained()
    elif kind == "batch":
        s["batch"] = fls.batch_c4(seed, case["segments"], case["log2_min"], case["log2_max"])
        s["tune"] = fls.tune(case["tile_vectors"], 256, fls.SCHED_DYNAMIC if case["dynamic"] else fls.SCHED_STATIC)
        s["counts"] = torch.zeros(case["segments"], dtype=torch.int64, device="cuda")
    elif kind == "train":
        s["feat"], s["label"], _ = selector.build_training_set(seed, case["samples"])
        s["mlp"] = selector.Mlp(seed)
        s["loss"] = torch.zeros(1, dtype=torch.float32, device="cuda")
    else:
        raise ValueError(kind)
    return s


# ----------------------------------------------------------------------- run
def run(s):
    case = s["case"]
    return RUN[case["kind"]](s, case)


def _run_q11(s, case):
    return fls.query_q11(*s["cols"], case["rows"], pred_load=case["pred_load"], d_out=s["out"], sync=False)


def _run_star(s, case):
    q, n = case["query"], case["rows"]
    if q == "q21_pht":
        return fls.query_q21_pht(*s["cols"], n, s["pht"], d_out=s["out"])
    call = {"q21": fls.query_q21, "q31": fls.query_q31, "q41": fls.query_q41}[q]
    return call(*s["cols"], n, s["dims"], s["ws"], d_out=s["out"])


def _run_unpack(s, case):
    if not case["checksum"]:
        fls.unpack_global(s["words"], s["out"], s["n_vec"], case["bw"])
        return s["out"]
    fls.unpack_checksum(s["words"], s["out"], case["values"], case["bw"], s["checksum"])
    return s["out"], s["checksum"][:1]


def _run_decode(s, case):
    col = s["col"]
    if case["via"] == "column":
        order = fls.ORDER_ROWS if case["order"] == "rows" else fls.ORDER_STORED
        return fls.decode_column(col, order=order, out=s["out"])
    if case["scheme"] == "delta":
        fls.delta_decode(col.words, col.vmeta, col.bases, s["n_vec"], s["out"])
    elif case["scheme"] == "rle":
        fls.rle_decode(col.words, col.vmeta, col.aux, col.bases, s["n_vec"], s["out"])
    else:
        selector.mixed_decode(col, out=s["out"])
    return s["out"]


def _run_encode(s, case):
    x, n, scheme = s["x"], case["rows"], case["scheme"]
    if scheme == "bitpack":
        return fls.pack_column_device(x, n, BITS_OF[case["data"]], transposed=True)
    if scheme == "delta":
        return fls.delta_encode_device(x, n)
    if scheme == "rle":
        return fls.rle_encode_device(x, n)
    if scheme == "exhaustive":
        selector.mixed_encode_exhaustive(x, n, s["ws"])
    else:
        s["selector"].encode(x, n, s["ws"])
    c = s["ws"].column(n)  # reads the encoded size, as a caller that stores the column does
    return c.words, c.vmeta, c.aux


def _run_batch(s, case):
    s["batch"].run(s["tune"], s["counts"])
    return s["counts"]


def _run_train(s, case):
    mlp = s["mlp"]
    s["loss"].zero_()
    mlp.accumulate_grad(s["feat"], s["label"], loss=s["loss"])
    mlp.adam()
    return mlp.w, mlp.m, mlp.v, s["loss"]


RUN = {"q11": _run_q11, "star": _run_star, "unpack": _run_unpack, "decode": _run_decode, "encode": _run_encode,
       "batch": _run_batch, "train": _run_train}


# ---------------------------------------------------------------------- work
# Encoded bits per value of the columns above, metadata apart.
DATA_BITS = {"quantities": 6.0, "prices": 24.0, "orderkeys": 1.0, "timestamps": 4.0, "runs": 1.0 + 16.0 / 8.0,
             "families": 12.0}


def _encoded_bytes(scheme, data, n):
    nv = selector.n_vectors(n)
    bits = DATA_BITS[data]
    if scheme == "rle" and data == "orderkeys":
        bits = 1.0 + 10.0 / 4.0
    if scheme in ("mixed", "exhaustive", "learned") and data == "orderkeys":
        bits = 1.0
    meta = {"bitpack": 0, "delta": 136, "rle": 144}.get(scheme, 16 + (128 if data in ("orderkeys", "runs") else 0))
    return n * bits / 8 + nv * meta


def work(case):
    kind = case["kind"]
    if kind == "q11":
        n = case["rows"]
        nv = selector.n_vectors(n)
        return {"bytes": n * 34 / 8 + nv * (136 if case["columns"] == "ssb" else 4 * 16 + 128), "flops": 0}
    if kind == "star":
        bits = {"q31": 12 + 20 + 16 + 24, "q41": 12 + 20 + 16 + 20 + 24 + 16}.get(case["query"], 12 + 16 + 20 + 24)
        return {"bytes": case["rows"] * bits / 8, "flops": 0}
    if kind == "unpack":
        n = selector.n_vectors(case["values"]) * VECTOR
        return {"bytes": n * (case["bw"] / 8 + 4), "flops": 0}
    if kind == "decode":
        return {"bytes": _encoded_bytes(case["scheme"], case["data"], case["rows"]) + 4 * case["rows"], "flops": 0}
    if kind == "encode":
        return {"bytes": _encoded_bytes(case["scheme"], case["data"], case["rows"]) + 4 * case["rows"], "flops": 0}
    if kind == "batch":
        # a segment is 40 % bit-packed, 30 % delta, 30 % RLE at a width of
        # U{1..32} bits, its length uniform in its octave; long delta segments
        # hold fewer bits a value (their sum stays below 2^32)
        octaves = range(case["log2_min"], case["log2_max"])
        n = sum(1.5 * 2 ** e for e in octaves) / len(octaves) * case["segments"]
        delta = min(16.5, max(1.0, 32.0 - case["log2_max"] + 0.5))
        bits = 0.4 * 16.5 + 0.3 * (delta + 8 * 136 / 1024) + 0.3 * (1 + 16.5 / 8 + 8 * 144 / 1024)
        return {"bytes": n * bits / 8, "flops": 0}
    params = 16 * 64 + 64 * 64 + 64 * 40
    return {"bytes": case["samples"] * 65 + 7848 * 24, "flops": case["samples"] * params * 2 * 3}


# --------------------------------------------------------------------- exact
def exact(case, seed):
    """The training step in 64 bits; every other case returns whole numbers."""
    if case["kind"] != "train":
        return None
    feat, label, _ = selector.build_training_set(seed, case["samples"])
    x = feat.cpu().numpy().astype(np.float64)
    y = label.cpu().numpy().astype(np.int64)
    w = selector.Mlp.init_weights(seed).astype(np.float64)
    parts, at = [], 0
    for fi, fo in ((16, 64), (64, 64), (64, 40)):
        parts.append((w[at:at + fi * fo].reshape(fi, fo), w[at + fi * fo:at + fi * fo + fo]))
        at += fi * fo + fo
    (w1, b1), (w2, b2), (w3, b3) = parts
    h1 = np.maximum(x @ w1 + b1, 0.0)
    h2 = np.maximum(h1 @ w2 + b2, 0.0)
    z = h2 @ w3 + b3
    z -= z.max(axis=1, keepdims=True)
    p = np.exp(z)
    p /= p.sum(axis=1, keepdims=True)
    rows = np.arange(len(y))
    loss = -np.log(p[rows, y]).sum()
    p[rows, y] -= 1.0
    dz = p / len(y)
    dh2 = (dz @ w3.T) * (h2 > 0)
    dh1 = (dh2 @ w2.T) * (h1 > 0)
    g = np.concatenate([a.ravel() for a in (x.T @ dh1, dh1.sum(0), h1.T @ dh2, dh2.sum(0), h2.T @ dz, dz.sum(0))])
    lr, beta1, beta2, eps = 2e-3, 0.9, 0.999, 1e-8
    m, v = (1 - beta1) * g, (1 - beta2) * g * g
    step = lr * (m / (1 - beta1)) / (np.sqrt(v / (1 - beta2)) + eps)
    return w - step, m, v, np.array([loss])
