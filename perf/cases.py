"""The work that is timed when this framework's speed is looked at: the calls
that a retrieval server and its offline jobs make, through the public entry
points of `manta_amd`, with the sizes of the configurations in `bench.py` and
generic ones around them.

A case is a dict of plain values.  `kind` says which call it is:

  topk    Runtime.score_topk: fused scoring + top-k over packed q8 / q4 rows
  score   Runtime.score: the whole score matrix (a reranker's call)
  embed   Runtime.embed_pooled: gather -> projection -> masked mean -> normalize
  encode  Runtime.encoder_pooled: the encoder's forward, one or two blocks
  dense   manta_rocm_dense_topk: f32 / f16 vectors, the retrieval evaluation

`prepare` makes the inputs on the GPU from the seed alone and binds them as a
server does at start-up; the outputs are buffers of the state, as a server
keeps them.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from manta_amd import _lib, rocm

_RT = None


def _runtime() -> rocm.Runtime:
    """One runtime (device + stream + workspace) per process."""
    global _RT
    if _RT is None:
        _RT = rocm.Runtime(0)
    return _RT


def listed():
    return [
        # a reranker's call: a few queries against the passages of a first
        # stage, every score wanted; the smallest work, all of it latency
        {"name": "rerank_scores_small", "kind": "score", "fmt": "q8", "op": "cosine", "nq": 8, "n": 1000, "d": 384},
        # one interactive query against a small q8 index, the quantized-query
        # formula (bench.py's config 0, one problem)
        {"name": "q8_dot_one_query", "kind": "topk", "fmt": "q8", "op": "dot", "quantized": True, "sets": 1, "nq": 1,
         "n": 65536, "d": 256, "k": 10},
        # 32 users, each with an index of their own (bench.py's headline)
        {"name": "q8_dot_32_indexes", "kind": "topk", "fmt": "q8", "op": "dot", "quantized": True, "sets": 32,
         "nq": 32, "n": 65536, "d": 256, "k": 10},
        # a handful of queries against a mid-sized index with the default
        # (reference) arithmetic; an odd row count
        {"name": "q8_cosine_few", "kind": "topk", "fmt": "q8", "op": "cosine", "quantized": False, "sets": 1, "nq": 4,
         "n": 262147, "d": 384, "k": 20},
        # one query against a large q4 index, candidates for a reranker
        {"name": "q4_dot_one_query", "kind": "topk", "fmt": "q4", "op": "dot", "quantized": False, "sets": 1, "nq": 1,
         "n": 1048576, "d": 384, "k": 100},
        # bench.py's config 2: a batch of queries against a large q4 index
        {"name": "q4_cosine_256", "kind": "topk", "fmt": "q4", "op": "cosine", "quantized": False, "sets": 1,
         "nq": 256, "n": 1048576, "d": 384, "k": 100},
        # bench.py's config 3: the l2 rerank stream, a long result list
        {"name": "q8_l2_smallest_1000", "kind": "topk", "fmt": "q8", "op": "l2_distance", "quantized": False,
         "sets": 1, "nq": 32, "n": 8388608, "d": 128, "k": 1000},
        # bench.py's config 4, second step: the largest work
        {"name": "q8_dot_1024", "kind": "topk", "fmt": "q8", "op": "dot", "quantized": True, "sets": 1, "nq": 1024,
         "n": 4194304, "d": 384, "k": 50},
        # bench.py's config 1: a batch of padded texts, f16 projection
        {"name": "embed_64x128", "kind": "embed", "b": 64, "t": 128, "d": 384, "e": 384, "proj": "f16",
         "prepared": False, "ragged": True},
        # bench.py's config 4, first step: a large batch, q8 projection bound once
        {"name": "embed_1024x64_q8", "kind": "embed", "b": 1024, "t": 64, "d": 384, "e": 384, "proj": "q8",
         "prepared": True, "ragged": False},
        # indexing a corpus with the encoder (bench.py's encoder workload), padded texts
        {"name": "encode_1024x64", "kind": "encode", "b": 1024, "t": 64, "d": 384, "h": 1536, "layers": 1},
        # retrieval evaluation: f32 vectors, a block of queries, the 100 best
        {"name": "dense_eval_f32", "kind": "dense", "dtype": "f32", "nq": 64, "n": 200000, "d": 384, "k": 100},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["topk", "topk", "topk", "topk", "score", "embed", "embed", "encode", "dense"])
    if kind in ("topk", "score"):
        fmt = rng.choice(["q8", "q8", "q4"])
        if fmt == "q4":
            d = rng.choice([128, 256, 384, 32 * rng.randint(1, 32)])
        else:
            d = rng.choice([128, 256, 384, 768, rng.randint(24, 1024)])
        op = rng.choice(["dot", "cosine", "l2_distance"])
        if kind == "score":
            nq = _log(rng, 1, 64)
            n = _log(rng, 100, min(1000000, 16000000 // nq))
            return {"kind": "score", "fmt": fmt, "op": op, "nq": nq, "n": n, "d": d}
        quantized = fmt == "q8" and op == "dot" and rng.random() < 0.5
        k = _log(rng, 1, 1000)
        if rng.random() < 0.2:  # an index per query
            sets = _log(rng, 2, 64)
            n = _log(rng, 1000, max(1000, 400000000 // (sets * d)))
            return {"kind": "topk", "fmt": fmt, "op": op, "quantized": quantized, "sets": sets, "nq": sets, "n": n,
                    "d": d, "k": min(k, n // 4)}
        nq = _log(rng, 1, 1024)
        n = _log(rng, 1000, max(1000, min(8388608, 800000000 // d, 400000000000 // (nq * d))))
        return {"kind": "topk", "fmt": fmt, "op": op, "quantized": quantized, "sets": 1, "nq": nq, "n": n, "d": d,
                "k": min(k, n // 4)}
    if kind == "embed":
        b = _log(rng, 1, 1024)
        t = _log(rng, 4, min(512, 131072 // b))
        d, e = rng.choice([(384, 384), (384, 384), (256, 256), (128, 384), (768, 768), (384, 128), (200, 96)])
        prepared = d % 32 == 0 and e % 128 == 0 and rng.random() < 0.5
        return {"kind": "embed", "b": b, "t": t, "d": d, "e": e, "proj": rng.choice(["f16", "q8"]),
                "prepared": prepared, "ragged": rng.random() < 0.7}
    if kind == "encode":
        b = _log(rng, 1, 1024)
        t = _log(rng, 8, min(256, 65536 // b))
        d, h = rng.choice([(384, 1536), (384, 1536), (256, 1024), (128, 512), (96, 384)])
        return {"kind": "encode", "b": b, "t": t, "d": d, "h": h, "layers": rng.choice([1, 2])}
    d = rng.choice([128, 256, 384, 768, rng.randint(24, 1024)])
    nq = _log(rng, 1, 512)
    n = _log(rng, 1000, max(1000, min(500000, 10000000000 // (nq * d))))
    return {"kind": "dense", "dtype": rng.choice(["f32", "f32", "f16"]), "nq": nq, "n": n, "d": d,
            "k": min(_log(rng, 1, 1000), n // 4)}


# ------------------------------------------------------------------- inputs

VOCAB = 32000  # bench.py's


def _gen(seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return g


def _normal(g, shape, sigma=1.0, normalize=False):
    x = torch.randn(shape, generator=g, device=g.device)
    if sigma != 1.0:
        x *= sigma
    return x / x.norm(dim=-1, keepdim=True) if normalize else x


def _uniform(g, lo, hi, shape, dtype=torch.int32):
    return torch.randint(lo, hi, shape, generator=g, device=g.device, dtype=dtype)


def _row_chunks(n, d):
    step = max(1, (1 << 27) // d)
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _q8_rows(g, n, d, normalize):
    """int8 codes [n, d] and f32 row scales: round(x * 127 / maxabs(row))."""
    codes = torch.empty((n, d), dtype=torch.int8, device=g.device)
    scales = torch.empty((n,), dtype=torch.float32, device=g.device)
    for a, b in _row_chunks(n, d):
        x = _normal(g, (b - a, d), normalize=normalize)
        s = x.abs().amax(dim=1) / 127.0
        codes[a:b] = (x / s[:, None]).round_().clamp_(-127, 127)
        scales[a:b] = s
    return codes, scales


def _q4_rows(g, n, d):
    """Signed nibbles as int8 [n, d] and f16 scales of blocks of 32."""
    codes = torch.empty((n, d), dtype=torch.int8, device=g.device)
    scales = torch.empty((n, d // 32), dtype=torch.float16, device=g.device)
    for a, b in _row_chunks(n, d):
        x = _normal(g, (b - a, d), normalize=True).view(b - a, d // 32, 32)
        s = (x.abs().amax(dim=2) / 7.0).half()
        codes[a:b] = (x / s.float()[..., None]).round_().clamp_(-7, 7).view(b - a, d)
        scales[a:b] = s
    return codes, scales


def _lengths_mask(g, b, t, ragged):
    if not ragged:
        return torch.ones((b, t), dtype=torch.int32, device=g.device)
    lengths = _uniform(g, max(1, t // 8), t + 1, (b, 1))
    return (torch.arange(t, device=g.device)[None, :] < lengths).to(torch.int32)


def _inputs(case, seed):
    """The call's inputs as tensors, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("topk", "score"):
        nq, n, d, sets = case["nq"], case["n"], case["d"], case.get("sets", 1)
        plain = case["op"] == "l2_distance"  # l2 ranks rows of any length
        x = {"queries": _normal(g, (nq, d), normalize=not plain).half()}
        if case["fmt"] == "q8":
            x["codes"], x["scales"] = _q8_rows(g, sets * n, d, not plain)
        else:
            x["codes"], x["scales"] = _q4_rows(g, sets * n, d)
        return x
    if kind == "dense":
        docs = _normal(g, (case["n"], case["d"]), normalize=True)
        return {"docs": docs.half() if case["dtype"] == "f16" else docs,
                "queries": _normal(g, (case["nq"], case["d"]), normalize=True)}
    b, t, d = case["b"], case["t"], case["d"]
    x = {"tokens": _uniform(g, 0, VOCAB, (b, t))}
    if kind == "embed":
        e = case["e"]
        x["mask"] = _lengths_mask(g, b, t, case["ragged"])
        x["table"] = _normal(g, (VOCAB, d), 0.02).half()
        if case["proj"] == "q8":
            x["proj"] = _uniform(g, -127, 128, (d, e), torch.int8)
            x["scales"] = (0.5 + torch.rand((e,), generator=g, device=g.device)) / (127.0 * math.sqrt(d))
        else:
            x["proj"] = _normal(g, (d, e), 1.0 / math.sqrt(d)).half()
        return x
    h = case["h"]
    x["mask"] = _lengths_mask(g, b, t, True)
    x["table"] = _uniform(g, -127, 128, (VOCAB, d), torch.int8)
    x["table_scales"] = (0.5 + torch.rand((VOCAB,), generator=g, device=g.device)) * (0.5 / 127.0)
    x["weights"] = []
    for rows, cols in [(d, d), (d, d), (d, d), (d, d), (d, h), (h, d)]:
        codes = _uniform(g, -127, 128, (rows, cols), torch.int8)
        scales = (0.5 + torch.rand((cols,), generator=g, device=g.device)) / (127.0 * math.sqrt(rows))
        x["weights"].append((codes, scales))
    return x


# ------------------------------------------------------- the call and its state

class _Memory:
    """A device array of the framework as torch sees it."""

    def __init__(self, array, typestr):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": typestr, "data": (array.addr, False),
                                         "version": 3}


def _view(array, typestr):
    return torch.as_tensor(_Memory(array, typestr), device="cuda")


def _host(x):
    x = x.cpu()
    return (x.view(torch.int16).numpy().view(np.uint16)) if x.dtype == torch.float16 else x.numpy()


def prepare(case, seed):
    rt = _runtime()
    kind = case["kind"]
    x = _inputs(case, seed)
    s = {"case": case, "rt": rt}
    if kind in ("topk", "score"):
        sets, n, d, nq = case.get("sets", 1), case["n"], case["d"], case["nq"]
        if case["fmt"] == "q8":
            s["cands"] = rt.bind_q8(_host(x["codes"]).reshape(sets, n, d), _host(x["scales"]).reshape(sets, n))
        else:
            nib = x["codes"].view(torch.uint8) & 15
            packed = nib[:, 0::2] | (nib[:, 1::2] << 4)  # low nibble first
            s["cands"] = rt.bind_q4(_host(packed).reshape(sets, n, d // 2),
                                    _host(x["scales"]).reshape(sets, n, d // 32), d)
        s["queries"] = rt.to_device(_host(x["queries"]))
        if kind == "score":
            s["out"] = rt.empty((nq, n), np.float32)
            s["views"] = {"scores": _view(s["out"], "<f4")}
        else:
            s["out"] = (rt.empty((nq, case["k"]), np.int32), rt.empty((nq, case["k"]), np.float32), None)
            s["views"] = {"ids": _view(s["out"][0], "<i4"), "scores": _view(s["out"][1], "<f4")}
        return s
    if kind == "dense":
        s["docs"], s["queries"] = rt.to_device(_host(x["docs"])), rt.to_device(_host(x["queries"]))
        s["out"] = (rt.empty((case["nq"], case["k"]), np.int32), rt.empty((case["nq"], case["k"]), np.float32))
        s["views"] = {"ids": _view(s["out"][0], "<i4"), "scores": _view(s["out"][1], "<f4")}
        return s
    s["tokens"], s["mask"] = rt.to_device(_host(x["tokens"])), rt.to_device(_host(x["mask"]))
    s["table"] = rt.to_device(_host(x["table"]))
    if kind == "embed":
        s["proj"] = rt.to_device(_host(x["proj"]))
        s["scales"] = rt.to_device(_host(x["scales"])) if case["proj"] == "q8" else None
        if case["prepared"]:
            s["proj"] = rt.prepare_projection(s["proj"])
        s["out"] = rt.empty((case["b"], case["e"]), np.uint16)
    else:
        s["table_scales"] = rt.to_device(_host(x["table_scales"]))
        s["weights"] = [(rt.to_device(_host(c)), rt.to_device(_host(v))) for c, v in x["weights"]]
        s["out"] = rt.empty((case["b"], case["d"]), np.uint16)
    s["views"] = {"embeddings": _view(s["out"], "<f2")}
    return s


def run(s):
    case, rt = s["case"], s["rt"]
    kind = case["kind"]
    if kind == "topk":
        rt.score_topk(s["cands"], case["op"], s["queries"], case["k"], smallest=case["op"] == "l2_distance",
                      out=s["out"], quantized=case["quantized"])
    elif kind == "score":
        rt.score(s["cands"], case["op"], s["queries"], out=s["out"])
    elif kind == "embed":
        rt.embed_pooled(s["tokens"], s["mask"], s["table"], s["proj"], s["scales"], out=s["out"])
    elif kind == "encode":
        rt.encoder_pooled(s["tokens"], s["mask"], s["table"], s["table_scales"], s["weights"], out=s["out"],
                          layers=case["layers"])
    else:
        # the C entry point: Runtime.dense_topk allocates its outputs anew
        _lib.call("manta_rocm_dense_topk", rt.handle, s["docs"].ptr,
                  C.c_int(_lib.DENSE_F16 if case["dtype"] == "f16" else _lib.DENSE_F32), C.c_int64(case["n"]),
                  C.c_int64(case["d"]), s["queries"].ptr, C.c_int64(case["nq"]), C.c_int64(case["d"]),
                  C.c_int64(case["k"]), s["out"][0].ptr, s["out"][1].ptr)
    return s["views"]


# ------------------------------------------------------------ what it costs

def work(case):
    kind = case["kind"]
    if kind in ("topk", "score", "dense"):
        nq, n, d = case["nq"], case["n"], case["d"]
        pairs = nq * n
        if kind == "dense":
            rows, q = n * d * (2 if case["dtype"] == "f16" else 4), nq * d * 4
        else:
            rows = case.get("sets", 1) * n * (d + 4 if case["fmt"] == "q8" else d // 2 + d // 16)
            q = nq * d * 2
            pairs = pairs if case.get("sets", 1) == 1 else case["sets"] * n
        out = pairs * 4 if kind == "score" else nq * case["k"] * 8
        return {"bytes": rows + q + out, "flops": 2 * pairs * d}
    b, t, d = case["b"], case["t"], case["d"]
    tokens = b * t
    if kind == "embed":
        e = case["e"]
        proj = d * e * (2 if case["prepared"] or case["proj"] == "f16" else 1)
        return {"bytes": tokens * (8 + 2 * d) + proj + 2 * b * e, "flops": 2 * tokens * d * e}
    h = case["h"]
    return {"bytes": tokens * (8 + d + 4) + 4 * d * d + 2 * d * h + 2 * b * d,
            "flops": case["layers"] * (2 * tokens * (4 * d * d + 2 * d * h) + 4 * b * t * t * d)}


def tolerance(case):
    # scores and ids are exact by the library's contract: the reference's
    # operations in the reference's order, or integer sums and a fixed chain
    # of roundings
    if case["kind"] in ("topk", "score", "dense"):
        return "exact"
    # f16 outputs of f32 sums: another order of the sums moves a few of them
    # to the next f16 value (two of the library's kernels: 1.3e-5, largest 8e-4)
    if case["kind"] == "embed":
        return {"rel": 5e-5, "max": 4e-3}
    # f16 operands of the block's products; a change of rounding in one step
    # travels through those that follow (two blocks against 64 bits: 2.8e-4,
    # largest 1.4e-3)
    return {"rel": 1e-3, "max": 6e-3}


# ------------------------------------------------------------ in 64 bits

def _rows64(case, x, a, b):
    """Rows a..b of the candidates as the values they stand for: f32 products
    code * scale (the quantized-query formula takes the codes themselves)."""
    codes = x["codes"][a:b]
    if case.get("quantized"):
        return codes.double()
    if case["fmt"] == "q8":
        return (codes.float() * x["scales"][a:b, None]).double()
    blocks = codes.view(b - a, -1, 32).float() * x["scales"][a:b].float()[..., None]
    return blocks.view(b - a, -1).double()


def _scores64(case, x, q, a, b):
    """Scores of the queries q [nq, d] against rows a..b."""
    rows = _rows64(case, x, a, b)
    dots = q @ rows.t().contiguous()
    if case.get("quantized"):  # codes round(q * 127 / qmax), qmax = 1 for unit queries
        return dots * x["scales"][a:b].double() / 127.0
    if case["op"] == "dot":
        return dots
    if case["op"] == "cosine":
        return dots / (q.norm(dim=1, keepdim=True) * rows.norm(dim=1)[None, :])
    d2 = (q * q).sum(1, keepdim=True) + (rows * rows).sum(1)[None, :] - 2.0 * dots
    return d2.clamp_(min=0).sqrt()


def _best(scores, k, smallest, best):
    """The k best values so far, best first."""
    if best is not None:
        scores = torch.cat([best, scores], dim=1)
    return scores.topk(min(k, scores.shape[1]), dim=1, largest=not smallest, sorted=True).values


def _layernorm64(x):
    x = x - x.mean(dim=-1, keepdim=True)
    return x / (x.square().mean(dim=-1, keepdim=True) + 1e-5).sqrt()


def _unit64(x):
    n = x.norm(dim=-1, keepdim=True)
    return torch.where(n > 0, x / n.clamp(min=1e-300), x)


def _mean64(x, mask):
    m = mask.double()[..., None]
    return (x * m).sum(dim=1) / m.sum(dim=1).clamp(min=1)


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("topk", "score", "dense"):
        n, d, nq = case["n"], case["d"], case["nq"]
        q = x["queries"].double()
        if case.get("quantized"):
            q = (q * 127.0).round().clamp(-127, 127)
        smallest = case.get("op") == "l2_distance"
        sets = case.get("sets", 1)
        parts = []
        step = max(1, (1 << 27) // max(d, nq))
        for s in range(sets):
            qs = q if sets == 1 else q[s:s + 1]
            best, whole = None, []
            for a in range(0, n, step):
                b = min(n, a + step)
                if kind == "dense":
                    got = qs @ x["docs"][a:b].double().t().contiguous()
                else:
                    got = _scores64(case, x, qs, s * n + a, s * n + b)
                if kind == "score":
                    whole.append(got)
                else:
                    best = _best(got, case["k"], smallest, best)
            parts.append(torch.cat(whole, dim=1) if kind == "score" else best)
        scores = torch.cat(parts, dim=0)
        return {"scores": scores} if kind == "score" else {"ids": None, "scores": scores}
    tokens = x["tokens"].long()
    if kind == "embed":
        proj = x["proj"].double()
        if case["proj"] == "q8":
            proj = proj * x["scales"].double()[None, :]
        y = x["table"].double()[tokens] @ proj
        return {"embeddings": _unit64(_mean64(y, x["mask"]))}
    w = [c.double() * v.double()[None, :] for c, v in x["weights"]]
    y = x["table"].double()[tokens] * x["table_scales"].double()[tokens][..., None]
    for _ in range(case["layers"]):
        qq, kk, vv = y @ w[0], y @ w[1], y @ w[2]
        att = torch.softmax(torch.matmul(qq, kk.transpose(1, 2).contiguous()), dim=-1)
        hid = _layernorm64(torch.matmul(att, vv) @ w[3] + y)
        up = hid @ w[4]
        up = 0.5 * up * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (up + 0.044715 * up ** 3)))
        y = _layernorm64(up @ w[5] + hid)
    return {"embeddings": _mean64(_unit64(y), x["mask"])}
