"""Workloads by which the route library's speed is judged.

Each case is one call (or one bank update followed by a call) as a program
that routes over grafts makes it, through the package's public classes.
Inputs follow the distributions of ``graftrepository_amd.workloads``:
unit-norm Gaussian centroid rows, N(0, 1) route keys, ragged node lengths.
They are drawn on the GPU from the seed and handed to the bank constructors
as the host arrays those take.

Every result is defined bit for bit (fp64 laws in a fixed order, rounded
once to fp32; ties go to the lowest node id), so the tolerance is exact.
``exact`` gives the scores in 64 bits.
"""

from __future__ import annotations

import math

import torch  # before the package: both then share one HIP runtime

import numpy as np

from graftrepository_amd import GqaNodeBank, MlaNodeBank
from graftrepository_amd.grm_hip_router import HipGQARouteSidecar, HipMLARouteSidecar
from graftrepository_amd.store_route import DeviceRouteStore

DEV = "cuda"
KINDS = ("turn", "doc", "digest", "era", "fact", "task_state", "recall", "cull_span")
FILTER_KINDS = ("turn", "doc")
VOCAB = 1000          # lexical keys in use over a store
QUERY_WORDS = 3       # lexical keys of a store query and of an indexed node


def listed():
    return [
        # A young session: a bank of ten thousand latent centroids, the
        # query straight from the forward pass, one route per step.
        dict(name="mla_single_10k", op="mla_single", nodes=10_000, dim=288, dtype="f32",
             host_query=False, k=3),
        # A long-lived arena at the size the project quotes its latency on.
        dict(name="mla_single_1m", op="mla_single", nodes=1_000_000, dim=288, dtype="f32",
             host_query=False, k=3),
        # The reference sidecar's own call: an fp32 bank, several host
        # queries at once; sizes that divide nothing.
        dict(name="mla_queries_100k", op="mla_queries", nodes=100_003, dim=280, queries=32, k=3),
        # A serving node that routes many sessions against one shared bank.
        dict(name="mla_batched_1m", op="mla_batched", nodes=1_000_000, dim=288, queries=256,
             query_dtype="bf16", k=8),
        # The same with the few requests of an ordinary step and a ragged bank.
        dict(name="mla_batched_150k", op="mla_batched", nodes=150_001, dim=200, queries=37,
             query_dtype="f32", k=5),
        # Prefill hands over its latent block; the key is formed on the GPU.
        dict(name="mla_latent_100k", op="mla_latent", nodes=100_000, dim=288, tokens=512, k=3),
        # An arena epoch: one percent of the nodes leave and as many come,
        # then the next route.
        dict(name="mla_churn_100k", op="mla_churn", nodes=100_000, dim=288, churn=1_000, k=3),
        # Decode over ragged per-token keys: four routing layers folded into
        # the head axes, one query token.
        dict(name="gqa_decode_512", op="gqa", nodes=512, lo=16, hi=512, kv=32, heads=128, hd=128,
             dtype="bf16", queries=1, tokens=1, k=3),
        # Prefill over such a bank: the prompt's last 64 tokens as the query.
        dict(name="gqa_prompt_256", op="gqa", nodes=256, lo=16, hi=512, kv=32, heads=128, hd=128,
             dtype="bf16", queries=1, tokens=64, k=3),
        # The reference arena's dense zero-padded fp32 hand-over, host query.
        dict(name="gqa_dense_f32_128", op="gqa_dense", nodes=128, key_tokens=251, kv=8, heads=32,
             hd=128, queries=1, tokens=4, k=3),
        # Packed INT8 grafts, the concurrent sessions' queries in one call.
        dict(name="gqa_int8_4000", op="gqa_int8", nodes=4_000, median=256, kv=8, heads=32, hd=128,
             queries=16, tokens=1, k=5),
        # The store's own route: lexical bonus and a kind filter.
        dict(name="store_100k", op="store", nodes=100_000, dim=288, k=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, hi=576):
    """A latent width: mostly a multiple of 32, sometimes any number."""
    d = _log(rng, 64, hi)
    return d if rng.random() < 0.3 else max(64, d // 32 * 32)


def draw(rng):
    op = rng.choice(["mla_single", "mla_single", "mla_queries", "mla_batched", "mla_batched",
                     "mla_latent", "mla_churn", "gqa", "gqa", "gqa_prompt", "gqa_dense",
                     "gqa_int8", "store"])
    k = rng.randint(1, 16)
    if op == "mla_single":
        dim, dtype = _dim(rng), rng.choice(["f32", "bf16"])
        return dict(op=op, nodes=min(_log(rng, 1_000, 1_000_000), 288_000_000 // dim), dim=dim,
                    dtype=dtype, host_query=rng.random() < 0.5, k=k)
    if op == "mla_queries":
        return dict(op=op, nodes=_log(rng, 1_000, 200_000), dim=_dim(rng),
                    queries=_log(rng, 2, 64), k=k)
    if op == "mla_batched":
        dim, queries = _dim(rng), _log(rng, 4, 256)
        nodes = min(_log(rng, 5_000, 1_000_000), 288_000_000 // dim,
                    256 * 288_000_000 // (dim * queries))
        return dict(op=op, nodes=nodes, dim=dim, queries=queries,
                    query_dtype=rng.choice(["bf16", "f32"]), k=k)
    if op == "mla_latent":
        return dict(op=op, nodes=_log(rng, 1_000, 300_000), dim=_dim(rng),
                    tokens=_log(rng, 8, 4096), k=k)
    if op == "mla_churn":
        nodes = _log(rng, 2_000, 200_000)
        return dict(op=op, nodes=nodes, dim=_dim(rng), churn=max(1, nodes // rng.randint(50, 400)),
                    k=k)
    if op in ("gqa", "gqa_prompt"):
        hd, kv = rng.choice([64, 128, 128, 256]), rng.choice([2, 4, 8, 16, 32])
        group = rng.choice([1, 2, 4, 4, 8])
        prompt = op == "gqa_prompt"
        queries = 1 if prompt else _log(rng, 1, 8)
        tokens = _log(rng, 8, 96) if prompt else rng.choice([1, 1, 2, 3, 4])
        hi = _log(rng, 64, 600)
        # at most half a billion key values, and 70 G multiply-adds
        row = (hi + 32) // 2 * kv * hd
        nodes = min(_log(rng, 24, 4_000), 500_000_000 // row,
                    70_000_000_000 // (row * group * queries * tokens))
        return dict(op="gqa", nodes=max(24, nodes), lo=rng.randint(1, 32), hi=hi, kv=kv,
                    heads=kv * group, hd=hd, dtype=rng.choice(["bf16", "f16"]), queries=queries,
                    tokens=tokens, k=k)
    if op == "gqa_dense":
        kv, hd = rng.choice([2, 4, 8]), rng.choice([64, 128, 256])
        return dict(op=op, nodes=_log(rng, 24, 256), key_tokens=_log(rng, 32, 512), kv=kv,
                    heads=kv * rng.choice([1, 2, 4, 7]), hd=hd, queries=_log(rng, 1, 6),
                    tokens=rng.choice([1, 2, 4, 5]), k=k)
    if op == "gqa_int8":
        hd, queries, tokens = rng.choice([64, 128]), _log(rng, 1, 32), rng.choice([1, 1, 2])
        median = _log(rng, 48, 256)
        nodes = min(_log(rng, 200, 6_000), 1_024_000 // median,
                    1_024_000 * 128 * 16 // (median * hd * queries * tokens))
        return dict(op=op, nodes=nodes, median=median, kv=rng.choice([4, 8]), heads=32, hd=hd,
                    queries=queries, tokens=tokens, k=k)
    return dict(op="store", nodes=_log(rng, 2_000, 200_000), dim=_dim(rng), k=k)


# ------------------------------------------------------------------- inputs


def _gen(seed, part):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + part) % (1 << 63))
    return g


def _unit(n, d, seed, part):
    x = torch.randn((n, d), generator=_gen(seed, part), device=DEV)
    return x / x.norm(dim=1, keepdim=True)


def _bits(t):
    """bf16 or fp16 values as the uint16 patterns the banks take."""
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _mla_rows(case, seed):
    rows = _unit(case["nodes"], case["dim"], seed, 1)
    return rows.bfloat16() if case.get("dtype") == "bf16" or case["op"] == "mla_batched" else rows


def _mla_queries(case, seed):
    q = _unit(case.get("queries", 1), case["dim"], seed, 2)
    dtype = case.get("query_dtype", case.get("dtype", "f32"))
    return q.bfloat16() if dtype == "bf16" else q


def _latent(case, seed):
    # tokens about a common direction, as the latents of one passage are
    g = _gen(seed, 3)
    base = torch.randn((1, case["dim"]), generator=g, device=DEV)
    noise = torch.randn((case["tokens"], case["dim"]), generator=g, device=DEV)
    return (base + noise).half()


def _lengths(case, seed):
    rng = np.random.default_rng([int(seed), 4])
    if case["op"] == "gqa_int8":
        x = np.exp(rng.normal(math.log(case["median"]), 0.5, size=case["nodes"]))
        return np.clip(np.rint(x), 1, 4096).astype(np.int64)
    if case["op"] == "gqa_dense":
        return rng.integers(max(1, case["key_tokens"] // 16), case["key_tokens"] + 1,
                            size=case["nodes"])
    return rng.integers(case["lo"], case["hi"] + 1, size=case["nodes"])


def _offsets(lengths):
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)


def _gqa_keys(case, seed, tokens):
    """Keys of all nodes back to back, [rows, hd], as the bank stores them:
    (values,) or for INT8 (codes, scales)."""
    rows, hd = int(tokens) * case["kv"], case["hd"]
    x = torch.randn((rows, hd), generator=_gen(seed, 5), device=DEV)
    if case["op"] == "gqa_int8":
        scale = (x.abs().amax(dim=1) / 127.0).half()
        scale[scale == 0] = 1.0
        codes = (x / scale.float()[:, None]).round().clamp(-128, 127).to(torch.int8)
        return codes, scale
    if case["op"] == "gqa_dense":
        return (x,)
    return (x.bfloat16() if case["dtype"] == "bf16" else x.half(),)


def _gqa_queries(case, seed):
    q = torch.randn((case["queries"], case["heads"], case["tokens"], case["hd"]),
                    generator=_gen(seed, 6), device=DEV)
    return q if case["op"] == "gqa_dense" else q.bfloat16()


def _words(case, seed):
    """Lexical keys of one node in a hundred, [nodes / 100, QUERY_WORDS]
    word numbers, and which nodes they are."""
    rng = np.random.default_rng([int(seed), 7])
    n = case["nodes"]
    who = np.sort(rng.choice(n, size=max(1, n // 100), replace=False))
    first = rng.integers(0, VOCAB, size=who.size)
    words = (first[:, None] + np.array([0, 131, 577])) % VOCAB
    kinds = rng.integers(0, len(KINDS), size=n)
    query = (int(words[0, 0]), int(words[0, 1]), int(rng.integers(0, VOCAB)))
    if query[2] in query[:2]:
        query = (query[0], query[1], (query[2] + 7) % VOCAB)
    return who, words, kinds, query


def prepare(case, seed):
    op, case = case["op"], dict(case)
    if op == "mla_single":
        rows, q = _mla_rows(case, seed), _mla_queries(case, seed)
        bits = case["dtype"] == "bf16"
        bank = MlaNodeBank(_bits(rows) if bits else rows.cpu().numpy(), dtype=case["dtype"])
        if case["host_query"]:
            q = _bits(q) if bits else q.cpu().numpy()
        return dict(case, bank=bank, q=q)
    if op == "mla_queries":
        bank = HipMLARouteSidecar().create_bank(_mla_rows(case, seed).cpu().numpy())
        return dict(case, bank=bank, q=_mla_queries(case, seed).cpu().numpy())
    if op == "mla_batched":
        bank = MlaNodeBank(_bits(_mla_rows(case, seed)), dtype="bf16")
        return dict(case, bank=bank, q=_mla_queries(case, seed))
    if op == "mla_latent":
        bank = MlaNodeBank(_mla_rows(case, seed).cpu().numpy())
        return dict(case, bank=bank, latent=_latent(case, seed))
    if op == "mla_churn":
        rows = _mla_rows(case, seed).cpu().numpy()
        ids = np.random.default_rng([int(seed), 8]).choice(case["nodes"], size=case["churn"],
                                                           replace=False).astype(np.uint64)
        fresh = _unit(case["churn"], case["dim"], seed, 9).cpu().numpy()
        return dict(case, bank=MlaNodeBank(rows), q=_mla_queries(case, seed), ids=ids, rows=fresh)
    if op == "gqa":
        lengths = _lengths(case, seed)
        keys, = _gqa_keys(case, seed, lengths.sum())
        bank = GqaNodeBank(_bits(keys), _offsets(lengths), kv_heads=case["kv"],
                           head_dim=case["hd"], dtype=case["dtype"])
        return dict(case, bank=bank, q=_gqa_queries(case, seed))
    if op == "gqa_dense":
        bank = HipGQARouteSidecar().create_bank(_dense(case, seed).cpu().numpy())
        return dict(case, bank=bank, q=_gqa_queries(case, seed).cpu().numpy())
    if op == "gqa_int8":
        lengths = _lengths(case, seed)
        codes, scales = _gqa_keys(case, seed, lengths.sum())
        bank = GqaNodeBank(codes.cpu().numpy(), _offsets(lengths), kv_heads=case["kv"],
                           head_dim=case["hd"], dtype="i8", scales=_bits(scales),
                           scale_dtype="f16", group_size=case["hd"])
        return dict(case, bank=bank, q=_gqa_queries(case, seed))
    who, words, kinds, query = _words(case, seed)
    lex = [()] * case["nodes"]
    for i, w in zip(who, words):
        lex[int(i)] = ["w%d" % x for x in w]
    store = DeviceRouteStore(case["dim"], capacity=case["nodes"])
    store.set_routes(np.arange(case["nodes"], dtype=np.uint64),
                     _mla_rows(case, seed).cpu().numpy(), lex,
                     [(KINDS[j], "", "", "") for j in kinds])
    return dict(case, bank=store, q=_mla_queries(case, seed)[0].cpu().numpy(),
                words=["w%d" % x for x in query])


def _dense(case, seed):
    """[nodes, kv, key_tokens, hd], zero past each node's length."""
    lengths = _lengths(case, seed)
    x, = _gqa_keys(case, seed, case["nodes"] * case["key_tokens"])
    x = x.view(case["nodes"], case["kv"], case["key_tokens"], case["hd"])
    keep = (torch.arange(case["key_tokens"], device=DEV)[None]
            < torch.from_numpy(lengths).to(DEV)[:, None])
    return x * keep[:, None, :, None]


# --------------------------------------------------------------------- pass


def run(state):
    op, bank, k = state["op"], state["bank"], state["k"]
    if op == "mla_single" and state["host_query"]:
        r = bank.route(state["q"], k, timed=False)
    elif op in ("mla_single", "mla_batched"):
        q = state["q"]
        r = bank.route(q, k, on_device=True, query_count=q.shape[0], timed=False,
                       query_dtype="bf16" if q.dtype == torch.bfloat16 else "f32")
    elif op in ("mla_queries", "gqa_dense"):
        ids, _ = bank.route_topk(state["q"], topk=k)
        return {"ids": ids.view(np.int64)}
    elif op == "mla_latent":
        r = bank.route_latent(state["latent"], state["tokens"], k, timed=False)
    elif op == "mla_churn":
        bank.evict(state["ids"])
        bank.append(state["rows"], state["ids"])
        r = bank.route(state["q"], k, on_device=True, query_count=1, timed=False)
    elif op in ("gqa", "gqa_int8"):
        r = bank.route(state["q"], k, on_device=True, query_dtype="bf16", timed=False)
    else:
        ids, scores = bank.route_scored(state["q"], state["words"], k, kinds=FILTER_KINDS)
        return {"ids": np.asarray(ids, np.int64), "scores": np.asarray(scores, np.float32)}
    return {"ids": r.ids.view(np.int64), "scores": r.scores}


# ------------------------------------------------------- bounds and results


def work(case):
    op, q = case["op"], case.get("queries", 1)
    out = 12 * q * case["k"]
    if op.startswith("gqa"):
        if op == "gqa":
            mean = (case["lo"] + case["hi"]) / 2
        elif op == "gqa_dense":
            mean = (max(1, case["key_tokens"] // 16) + case["key_tokens"]) / 2
        else:
            mean = case["median"] * math.exp(0.125)  # lognormal, sigma 0.5
        tokens = case["nodes"] * mean
        row = case["hd"] + 2 if op == "gqa_int8" else case["hd"] * (4 if op == "gqa_dense" else 2)
        query = q * case["heads"] * case["tokens"] * case["hd"] * (4 if op == "gqa_dense" else 2)
        return {"bytes": tokens * case["kv"] * row + query + out,
                "flops": 2.0 * q * case["heads"] * case["tokens"] * tokens * case["hd"]}
    two = op == "mla_batched" or case.get("dtype") == "bf16"
    size = 2 if two else 4
    bytes_ = case["nodes"] * (case["dim"] * size + 4) + q * case["dim"] * 4 + out
    flops = 2.0 * q * case["nodes"] * case["dim"]
    if op == "mla_latent":
        bytes_ += case["tokens"] * case["dim"] * 2
        flops += case["tokens"] * case["dim"]
    if op == "mla_churn":
        bytes_ += 2 * case["churn"] * case["dim"] * 4
    if op == "store":
        bytes_ += 8 * case["nodes"]  # the nodes' filter bits
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # fp64 sums in a fixed order, one rounding to fp32: every bit is given
    return "exact"


def _top(scores, k):
    return torch.sort(scores, dim=1, descending=True).values[:, :k].cpu()


def _mla_scores(rows, q):
    rows = rows.double()
    norm = rows.square().sum(dim=1).sqrt().float().double()
    out = []
    for one in q.double():
        out.append((rows * one).sum(dim=1) / (one.square().sum().sqrt() * norm + 1e-8))
    return torch.stack(out)


def _gqa_scores(blocks, q, kv):
    """blocks: per node [kv, L, hd] in fp64; q [Q, H, Qt, hd]."""
    nq, heads, qt, hd = q.shape
    cols = q.double().view(nq, kv, heads // kv, qt, hd).transpose(0, 1).reshape(kv, -1, hd)
    out = []
    for b in blocks:
        dot = torch.matmul(cols.contiguous(), b.transpose(1, 2).contiguous()).abs()
        best = dot.amax(dim=2).view(kv, nq, heads // kv, qt).amax(dim=3) / math.sqrt(hd)
        out.append(best.sum(dim=(0, 2)) / heads)
    return torch.stack(out, dim=1)


def exact(case, seed):
    op, k = case["op"], case["k"]
    if op in ("mla_queries", "gqa_dense"):
        return None  # whole numbers only
    if op.startswith("gqa"):
        lengths = _lengths(case, seed)
        keys = _gqa_keys(case, seed, lengths.sum())
        values = (keys[0].float() * keys[1].float()[:, None]).half() if len(keys) == 2 else keys[0]
        ends = np.cumsum(lengths) * case["kv"]

        def blocks():
            for n, end in zip(lengths, ends):
                rows = values[int(end - n * case["kv"]):int(end)]
                yield rows.view(case["kv"], int(n), case["hd"]).double()

        return {"ids": None, "scores": _top(_gqa_scores(blocks(), _gqa_queries(case, seed),
                                                        case["kv"]), k)}
    rows = _mla_rows(case, seed)
    if op == "mla_latent":
        mean = _latent(case, seed).double().mean(dim=0)
        q = (mean / (mean.norm() + 1e-8))[None]
    else:
        q = _mla_queries(case, seed)
    if op == "mla_churn":
        ids = np.random.default_rng([int(seed), 8]).choice(case["nodes"], size=case["churn"],
                                                           replace=False)
        rows = rows.clone()
        rows[torch.from_numpy(ids).to(DEV)] = _unit(case["churn"], case["dim"], seed, 9)
    scores = _mla_scores(rows, q)
    if op == "store":
        who, words, kinds, query = _words(case, seed)
        hits = np.zeros(case["nodes"])
        hits[who] = np.isin(words, query).sum(axis=1)
        scores = scores + torch.from_numpy(hits / QUERY_WORDS).to(DEV)
        ok = torch.from_numpy(np.isin(kinds, [KINDS.index(x) for x in FILTER_KINDS])).to(DEV)
        scores = torch.where(ok[None], scores, torch.full_like(scores, -math.inf))
        return {"ids": None, "scores": _top(scores, k)[0]}
    return {"ids": None, "scores": _top(scores, k)}
