"""The calls whose speed counts: what users of this operator have it do, over the range they do it in.

A case is a plain dict; ``kind`` says which public entry point it goes through and what it stands for:

* ``dense``   attention() without a mask or causal only: encoders, pre-training on unpacked sequences
* ``doc``     attention() with document ids: pre-training on packed documents, also against a longer key range
* ``local``   attention() with a sliding window or a bidirectional prefix
* ``block``   attention() with a block map
* ``packed``  attention_varlen(), queries and keys with the same boundaries: fine-tuning on sequences of mixed length
* ``chunk``   attention_varlen(), each sequence's queries are the tail of its keys: chunked prefill, mixed decoding
* ``decode``  attention() of one or a few new tokens against a cache of keys and values

``mode`` is "fb" (a training step's forward and backward) or "fwd" (inference, under no_grad).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "triton-flash-attention-with-flexible-masks_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from flash_mi355 import SCORE_FUNC_MODE0_NOPE, SCORE_FUNC_MODE1_DOC, attention, attention_varlen, workloads  # noqa: E402

_TORCH = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def _case(kind, mode, dtype, B, H, Hk, M, N, D, causal=True, layout="bhld", **more):
    return dict(kind=kind, mode=mode, dtype=dtype, B=B, H=H, Hk=Hk, M=M, N=N, D=D, causal=causal, layout=layout, **more)


def listed():
    named = [
        # a small fp32 problem with documents, forward and backward: gradient checks, small models, the first configuration of the benchmark
        ("small_fp32_doc", _case("doc", "fb", "fp32", 2, 4, 4, 512, 512, 64, doc="uniform", doc_a=32, doc_b=256, glob=0.05, ids="int64")),
        # one short prompt of an odd length through a grouped-query model: the latency of a single call
        ("short_prompt", _case("dense", "fwd", "bf16", 1, 32, 8, 333, 333, 128, layout="blhd")),
        # an encoder's training step: no mask, short heads
        ("plain_2k", _case("dense", "fb", "bf16", 4, 16, 16, 2048, 2048, 64, causal=False)),
        # packed documents at an ordinary context length, a tenth of the tokens global
        ("doc_4k", _case("doc", "fb", "bf16", 2, 32, 32, 4096, 4096, 128, doc="uniform", doc_a=128, doc_b=1024, glob=0.10, ids="int32")),
        # the headline: packed documents at 16K tokens
        ("doc_16k", _case("doc", "fb", "bf16", 1, 32, 32, 16384, 16384, 128, doc="geometric", doc_a=512, doc_b=16, glob=0.02, ids="int32")),
        # a query block against a longer packed key range, fp16
        ("rect_doc", _case("doc", "fb", "fp16", 8, 8, 8, 1024, 8192, 128, doc="equal", doc_a=256, doc_b=256, glob=0.05, ids="int32")),
        # the largest: long-context training without documents
        ("causal_16k", _case("dense", "fb", "bf16", 1, 32, 32, 16384, 16384, 128)),
        # a sliding window of 1024 keys over a long context
        ("window_16k", _case("local", "fb", "bf16", 1, 32, 32, 16384, 16384, 128, window=1024, prefix=0)),
        # block-sparse training: the diagonal and a quarter of the other blocks
        ("block_16k", _case("block", "fb", "bf16", 1, 32, 32, 16384, 16384, 128, density=0.25)),
        # fine-tuning on a packed batch of sequences of odd lengths, grouped-query heads
        ("packed_train", _case("packed", "fb", "bf16", 1, 32, 8, 0, 0, 128, layout="thd", seqs=24, q_lo=64, q_hi=1200, k_lo=0, k_hi=0)),
        # chunked prefill of a serving batch: up to 128 new tokens each on top of some two thousand cached ones
        ("chunked_prefill", _case("chunk", "fwd", "bf16", 1, 32, 8, 0, 0, 128, layout="thd", seqs=32, q_lo=17, q_hi=128, k_lo=500, k_hi=3500)),
        # one decoding step of a serving batch against its cache
        ("decode", _case("decode", "fwd", "bf16", 16, 32, 8, 1, 6001, 128, layout="cache", capacity=8192)),
    ]
    return [dict(c, name=name) for name, c in named]


# The largest listed case's work; a drawn case stays below it (fp32 products cost sixteen times a 16-bit one's).
_MOST_FLOPS = 3.5 * 4 * 32 * 128 * 16384 * 16384 / 2
_MOST_FLOPS_FP32 = _MOST_FLOPS / 30
_MOST_BYTES = 2.5e9


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(("dense", "dense", "doc", "doc", "doc", "local", "block", "packed", "packed", "chunk", "decode", "decode"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    D = rng.choice((64, 128, 128))
    Hk = rng.choice((2, 4, 8, 8, 16))
    H = Hk * rng.choice((1, 1, 2, 4))
    mode = rng.choice(("fb", "fb", "fwd"))
    layout = rng.choice(("bhld", "blhd"))
    B = rng.choice((1, 1, 2, 3, 4, 8))
    if kind == "dense":
        L = _log(rng, 64, 16384)
        if rng.random() < 0.25 and L <= 4096:
            dtype, D = "fp32", 64
        return _case(kind, mode, dtype, B, H, Hk, L, L, D, causal=rng.random() < 0.7, layout=layout)
    if kind == "doc":
        L = _log(rng, 256, 16384)
        if rng.random() < 0.25 and L <= 4096:
            dtype, D, Hk = "fp32", 64, H
        M = L if rng.random() < 0.75 else max(32, int(L * rng.uniform(0.1, 0.6)))
        a = _log(rng, 48, 1024)
        doc, a, b = rng.choice((("uniform", max(16, a // 2), 2 * a), ("geometric", a, 16)))
        return _case(kind, mode, dtype, B, H, Hk, M, L, D, layout=layout, doc=doc, doc_a=a, doc_b=b,
                     glob=rng.choice((0.0, 0.02, 0.05, 0.10)), ids=rng.choice(("int32", "int64")))
    if kind == "local":
        L = _log(rng, 512, 16384)
        w = _log(rng, 64, max(65, L // 4))
        prefix = rng.random() < 0.3
        return _case(kind, mode, dtype, B, H, Hk, L, L, D, layout=layout, window=0 if prefix else w, prefix=w if prefix else 0)
    if kind == "block":
        L = _log(rng, 1024, 16384)
        return _case(kind, mode, dtype, B, H, Hk, L, L, D, layout=layout, density=round(rng.uniform(0.1, 0.5), 2))
    if kind == "packed":
        hi = _log(rng, 48, 4096)
        return _case(kind, mode, dtype, 1, H, Hk, 0, 0, D, layout="thd", seqs=_log(rng, 1, max(2, 32768 // hi)), q_lo=max(1, hi // 16), q_hi=hi,
                     k_lo=0, k_hi=0)
    if kind == "chunk":
        k_hi = _log(rng, 128, 8192)
        q_hi = min(k_hi // 2, _log(rng, 1, 512))
        return _case(kind, "fwd", dtype, 1, H, Hk, 0, 0, D, layout="thd", seqs=_log(rng, 1, max(2, min(64, 65536 // k_hi))),
                     q_lo=max(1, q_hi // 8), q_hi=max(1, q_hi), k_lo=max(1, k_hi // 8), k_hi=k_hi)
    N = _log(rng, 100, 32768)
    B = max(1, min(32, _log(rng, 1, 64), 262144 // N))
    return _case("decode", "fwd", dtype, B, H, Hk, rng.choice((1, 1, 1, 2, 4, 8)), N, D, layout="cache", capacity=-(-N // 1024) * 1024)


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= (_MOST_FLOPS_FP32 if c["dtype"] == "fp32" else _MOST_FLOPS) and w["bytes"] <= _MOST_BYTES:
            return c


# -- what the inputs look like ----------------------------------------------------------------------------------------------
def _doc_ids(c, rng):
    """(eq [B, M], ek [B, N]) as numpy: documents packed over the keys, the queries are the last M tokens."""
    L = c["N"]
    rows = []
    for _ in range(c["B"]):
        if c["doc"] == "uniform":
            rows.append(workloads.doc_ids_uniform(rng, L, c["doc_a"], c["doc_b"], 0.0))
        elif c["doc"] == "geometric":
            rows.append(workloads.doc_ids_geometric(rng, L, c["doc_a"], c["doc_b"], 0.0))
        else:
            rows.append(-(np.arange(L) // c["doc_a"] + 1).astype(np.int32))
    own = np.stack(rows)
    g = rng.random(own.shape) < c["glob"]
    ids = np.where(g, 0, own).astype(np.int32)
    if c["M"] == c["N"]:
        return ids, ids
    return np.ascontiguousarray(ids[:, L - c["M"]:]), own   # a longer key range keeps its own ids


def _lengths(c, rng):
    """(query lengths, key lengths): the case's own, in an order of the seed's (the totals, and so the shapes, stay)."""
    of_case = np.random.default_rng([c["seqs"], c["q_hi"], c["k_hi"]])
    q = k = of_case.integers(c["q_lo"], c["q_hi"] + 1, c["seqs"])
    if c["k_hi"]:
        k = np.maximum(q, of_case.integers(c["k_lo"], c["k_hi"] + 1, c["seqs"]))
    order = rng.permutation(c["seqs"])
    return q[order], k[order]


def _block_map(c, rng):
    n = -(-c["M"] // 64)
    return (rng.random((1, 1, n, n)) < c["density"]) | np.eye(n, dtype=bool)[None, None]


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(_TORCH[dtype])


def _heads(gen, c, heads, length):
    """[B, heads, length, D] in the case's memory order."""
    if c["layout"] == "blhd":
        return _randn(gen, (c["B"], length, heads, c["D"]), c["dtype"]).transpose(1, 2)
    return _randn(gen, (c["B"], heads, length, c["D"]), c["dtype"])


def prepare(case, seed):
    c, rng = case, np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": c}
    if c["kind"] in ("packed", "chunk"):
        q_len, k_len = _lengths(c, rng)
        cu = [torch.from_numpy(np.concatenate([[0], np.cumsum(n)]).astype(np.int32)).cuda() for n in (q_len, k_len)]
        s["cu_q"], s["cu_k"] = cu[0], cu[1] if c["k_hi"] else None
        tq, tk = int(q_len.sum()), int(k_len.sum())
        shapes = [(tq, c["H"], c["D"]), (tk, c["Hk"], c["D"]), (tk, c["Hk"], c["D"])]
        s["qkv"] = [_randn(gen, n, c["dtype"]) for n in shapes]
        s["do"] = _randn(gen, shapes[0], c["dtype"])
    elif c["kind"] == "decode":
        s["qkv"] = [_randn(gen, (c["B"], c["H"], c["M"], c["D"]), c["dtype"])]
        for _ in range(2):   # the filled part of a cache with room for more
            s["qkv"].append(_randn(gen, (c["B"], c["Hk"], c["capacity"], c["D"]), c["dtype"])[:, :, :c["N"]])
    else:
        s["qkv"] = [_heads(gen, c, c["H"], c["M"]), _heads(gen, c, c["Hk"], c["N"]), _heads(gen, c, c["Hk"], c["N"])]
        s["do"] = _heads(gen, c, c["H"], c["M"])
        if c["kind"] == "doc":
            kind = torch.int64 if c["ids"] == "int64" else torch.int32
            eq, ek = _doc_ids(c, rng)
            s["eq"] = torch.from_numpy(eq).to("cuda", kind)[:, None].expand(c["B"], c["H"], c["M"])
            s["ek"] = torch.from_numpy(ek).to("cuda", kind)[:, None].expand(c["B"], c["H"], c["N"])
        elif c["kind"] == "block":
            s["block"] = torch.from_numpy(_block_map(c, rng)).cuda()
    if c["mode"] == "fb":
        s["qkv"] = [t.requires_grad_(True) for t in s["qkv"]]
    return s


# -- one pass ---------------------------------------------------------------------------------------------------------------
def _forward(s):
    c, (q, k, v) = s["case"], s["qkv"]
    if c["kind"] in ("packed", "chunk"):
        return attention_varlen(q, k, v, s["cu_q"], s["cu_k"], causal=c["causal"])
    if c["kind"] == "doc":
        return attention(q, k, v, c["causal"], None, s["eq"], s["ek"], SCORE_FUNC_MODE1_DOC)
    if c["kind"] == "block":
        return attention(q, k, v, c["causal"], block_mask=s["block"])
    if c["kind"] == "local":
        return attention(q, k, v, c["causal"], window=c["window"], prefix=c["prefix"])
    return attention(q, k, v, c["causal"], None, None, None, SCORE_FUNC_MODE0_NOPE)


def run(state):
    if state["case"]["mode"] == "fwd":
        with torch.no_grad():
            return {"o": _forward(state)}
    o = _forward(state)
    dq, dk, dv = torch.autograd.grad(o, state["qkv"], state["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


# -- what a pass cannot do without ------------------------------------------------------------------------------------------
def _causal_pairs(m, n):
    """Kept pairs of m rows against n >= m keys, aligned at the end."""
    return m * (n - m) + m * (m + 1) // 2


def _pairs(c):
    """(kept (row, key) pairs of one head over the whole batch, rows, keys); masks that depend on the seed as seed 0 makes them."""
    rng = np.random.default_rng(0)
    if c["kind"] in ("packed", "chunk"):
        q_len, k_len = _lengths(c, rng)
        pairs = sum(_causal_pairs(int(m), int(n)) if c["causal"] else int(m) * int(n) for m, n in zip(q_len, k_len))
        return pairs, int(q_len.sum()), int(k_len.sum())
    B, M, N = c["B"], c["M"], c["N"]
    if c["kind"] == "doc":
        pairs = 0
        for eq, ek in zip(*_doc_ids(c, rng)):
            pos = np.arange(M) + N - M
            order = np.argsort(ek, kind="stable")
            rank = np.empty(N, np.int64)      # how many keys of the same id lie before a key
            ids, first = np.unique(ek[order], return_index=True)
            rank[order] = np.arange(N) - first[np.searchsorted(ids, ek[order])]
            # a local row sits on its own key unless that key carries a document id of its own
            pairs += int(np.where(eq >= 0, pos + 1, rank[pos] + 1).sum())
        return pairs, B * M, B * N
    if c["kind"] == "local":
        pos = np.arange(M, dtype=np.int64) + 1
        seen = np.minimum(pos, c["window"]) if c["window"] else np.maximum(pos, min(c["prefix"], N))
        return B * int(seen.sum()), B * M, B * N
    if c["kind"] == "block":
        on, n = _block_map(c, rng)[0, 0], -(-M // 64)
        return B * int(np.tril(on, -1).sum() * 64 * 64 + n * (64 * 65 // 2)), B * M, B * N
    return B * (_causal_pairs(M, N) if c["causal"] else M * N), B * M, B * N


def work(case):
    pairs, rows, keys = _pairs(case)
    q, kv = rows * case["H"] * case["D"], 2 * keys * case["Hk"] * case["D"]
    elems = 2 * q + kv                       # q, k, v read, o written
    if case["mode"] == "fb":
        elems += 2 * q + kv                  # do read, dq, dk, dv written
    more = 0
    if case["kind"] == "doc":
        more = (rows + keys) * (8 if case["ids"] == "int64" else 4)
    elif case["kind"] == "block":
        more = (-(-case["M"] // 64)) ** 2
    return {"bytes": elems * _BYTES[case["dtype"]] + more, "flops": 4 * pairs * case["H"] * case["D"] * (3.5 if case["mode"] == "fb" else 1.0)}


def tolerance(case):
    # sums of products in fp32; the weights, the gradients of the scores and the results are rounded to the tensors' type
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}
