"""Performance cases of the scoring paths, through the entry points a program calls.

Every case names an operation and its sizes.  Corpora are seeded: documents of
uniform random length whose tokens are a random centroid plus noise,
L2-normalised, as maxsim_amd.synthetic makes them (here on the GPU, so that
they are quick to make); queries are perturbed tokens of a document.  Handles
are built once, as a serving program keeps them; a pass is one call with its
query in hand.

Operations:
  int8_search      int4 corpus, int8-quantised query, top-k: numpy in and out
                   (host) or device tensors on the current stream
  int8_scores      the same query against every document, the whole [B, N]
  fp32_search      int4 corpus, fp32 query, any reducer, top-k (numpy)
  rerank           int4 corpus, fp32 query, given candidates (numpy)
  residual_search  int4 prefix + int4 residual, fp32 query: candidates > 0 the
                   cascade, 0 every document fused (numpy)
  binary_search    sign corpus, fp32 query, top-k (numpy), with or without
                   per-token scales
  hamming_search   sign corpus, sign queries, top-k (device tensors)
  binres_search    sign prefix + int4 residual cascade, int8 query (device
                   tensors)
  pack             per-token int4 packing of embeddings that are on the GPU
"""
from __future__ import annotations

import numpy as np
import torch

from maxsim_amd import (
    Int4PackedDocs,
    PackedDocs,
    int4_maxsim,
    pack_int4_symmetric_device,
    topk_int4_maxsim,
    topk_maxsim,
)
from maxsim_amd._maxsim_hip import CudaInt4PackedDocs, CudaPackedDocs

DEV = "cuda"


def listed():
    return [
        # An interactive search over a small collection: one query, host
        # arrays in and out; latency and launches are what it costs.
        {"name": "int8_small_host", "op": "int8_search", "docs": 512, "lo": 32, "hi": 64, "batch": 1, "qt": 32,
         "k": 10, "host": True},
        # The headline: four queries against a page of 4,096 ragged documents,
        # everything on the device.
        {"name": "int8_search", "op": "int8_search", "docs": 4096, "lo": 64, "hi": 192, "batch": 4, "qt": 32,
         "k": 10, "host": False},
        # A large collection streamed from HBM for one query, a first stage
        # that keeps a hundred documents.
        {"name": "int8_large", "op": "int8_search", "docs": 65536, "lo": 64, "hi": 192, "batch": 1, "qt": 32,
         "k": 100, "host": False},
        # Full score rows (the caller fuses them with other signals): odd
        # document counts, very short to long documents, a query length that
        # is no multiple of a tile, more rows than one pass holds.
        {"name": "int8_scores_ragged", "op": "int8_scores", "docs": 3001, "lo": 1, "hi": 300, "batch": 7, "qt": 21},
        # Search on the unquantised query.
        {"name": "fp32_search", "op": "fp32_search", "docs": 4096, "lo": 64, "hi": 192, "dim": 128, "batch": 4,
         "qt": 32, "k": 10, "reducer": "maxsim"},
        # Second stage after another retriever: a given candidate list.
        {"name": "rerank", "op": "rerank", "docs": 4096, "lo": 64, "hi": 192, "dim": 128, "batch": 1, "qt": 32,
         "candidates": 500, "reducer": "maxsim"},
        # Higher-quality format: coarse pass, 512 candidates, fused rescoring.
        {"name": "residual_cascade", "op": "residual_search", "docs": 4096, "lo": 64, "hi": 192, "batch": 4, "qt": 32,
         "k": 10, "candidates": 512, "reducer": "maxsim"},
        # Visual-patch pages as signs, one fp32 query.
        {"name": "binary_search", "op": "binary_search", "docs": 10240, "lo": 256, "hi": 1024, "batch": 1, "qt": 32,
         "k": 10, "token_scale": False},
        # The same pages, a batch of 256 sign queries (offline evaluation).
        {"name": "hamming_batch", "op": "hamming_search", "docs": 10240, "lo": 256, "hi": 1024, "batch": 256, "qt": 32,
         "k": 10},
        # Sign prefix, int4 residual cascade.
        {"name": "binres_cascade", "op": "binres_search", "docs": 4096, "lo": 64, "hi": 192, "batch": 4, "qt": 32,
         "k": 10, "candidates": 512},
        # Wider embeddings and another reducer.
        {"name": "fp32_wide", "op": "fp32_search", "docs": 2000, "lo": 16, "hi": 200, "dim": 256, "batch": 2, "qt": 24,
         "k": 10, "reducer": "topk4"},
        # Index build of one ingestion batch.
        {"name": "pack", "op": "pack", "tokens": 65536, "dim": 128},
    ]


REDUCERS = ("maxsim", "weighted_maxsim", "topk2", "topk4", "smoothsim")
# Document lengths: passages, paragraphs, anything from one token up.
LENGTHS = ((32, 64), (64, 192), (1, 300), (17, 90))


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))

    op = rng.choice(["int8_search", "int8_search", "int8_scores", "fp32_search", "fp32_search", "rerank",
                     "residual_search", "binary_search", "hamming_search", "binres_search", "pack"])
    lo, hi = rng.choice(LENGTHS)
    case = {"op": op, "docs": log_int(200, 12000), "lo": lo, "hi": hi, "batch": log_int(1, 8), "qt": rng.randint(4, 48)}
    if op == "int8_search":
        case["docs"] = log_int(200, 65536)
        case["k"] = min(log_int(1, 100), case["docs"])
        case["host"] = rng.random() < 0.5
        if case["docs"] > 8192:
            case["batch"] = min(case["batch"], 4)
    elif op == "fp32_search":
        case["k"] = log_int(1, 32)
        case["dim"] = rng.choice([128, 128, 64, 200, 256])
        case["reducer"] = rng.choice(REDUCERS)
        case["batch"] = min(case["batch"], 4)
    elif op == "rerank":
        case["dim"] = rng.choice([128, 128, 96, 256])
        case["reducer"] = rng.choice(REDUCERS)
        case["candidates"] = min(log_int(16, 2000), case["docs"])
        case["batch"] = min(case["batch"], 4)
    elif op == "residual_search":
        case["batch"] = min(case["batch"], 4)
        case["k"] = log_int(1, 16)
        case["candidates"] = rng.choice([0, min(case["docs"], log_int(64, 1024))])
        case["reducer"] = rng.choice(REDUCERS)
    elif op == "binary_search":
        case["lo"], case["hi"] = rng.choice([(64, 192), (256, 1024), (1, 300)])
        case["batch"] = min(case["batch"], 4)
        case["k"] = log_int(1, 32)
        case["token_scale"] = rng.random() < 0.5
    elif op == "hamming_search":
        case["lo"], case["hi"] = rng.choice([(64, 192), (256, 1024), (1, 300)])
        case["docs"] = log_int(200, 10240)
        case["batch"] = log_int(1, 128)
        case["k"] = log_int(1, 32)
    elif op == "binres_search":
        case["docs"] = log_int(600, 8192)
        case["k"] = log_int(1, 16)
        case["candidates"] = log_int(64, 600)
        case["batch"] = min(case["batch"], 4)
    elif op == "pack":
        case = {"op": "pack", "tokens": log_int(1000, 262144), "dim": rng.choice([64, 128, 128, 256])}
    return case


# ------------------------------------------------------------------- inputs


def _generator(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + stream)
    return g


def _lengths(case, seed):
    rng = np.random.default_rng([int(seed), 17])
    return rng.integers(case["lo"], case["hi"] + 1, size=case["docs"]).astype(np.int64)


def _unit(x):
    return x / x.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _embedding_blocks(lens, dim, seed, block_docs=8192):
    """Unit tokens of the documents, in blocks of documents."""
    g = _generator(seed, 1)
    for first in range(0, len(lens), block_docs):
        n = torch.from_numpy(lens[first:first + block_docs]).to(DEV)
        centroids = torch.randn(len(n), dim, generator=g, device=DEV)
        x = torch.repeat_interleave(centroids, n, dim=0)
        x += 0.5 * torch.randn(x.shape, generator=g, device=DEV)
        yield _unit(x)


def _int4(x):
    """Symmetric per-token int4: (values int8 [T, dim], scales f32 [T])."""
    s = x.abs().amax(dim=1) / 7.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(x / s[:, None]), -7, 7).to(torch.int8), s


def _nibbles(v):
    """Two's-complement nibbles, even dim in the low half."""
    u = v.view(torch.uint8) & 15
    return u[:, 0::2] | (u[:, 1::2] << 4)


def _sign_bits(x):
    """Sign bits, bit j of byte j / 8, set for x >= 0."""
    b = (x >= 0).view(x.shape[0], -1, 8).to(torch.uint8)
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=x.device)
    return (b * w).sum(dim=2, dtype=torch.int64).to(torch.uint8)


def _corpus(case, seed, streams):
    """{"offsets", "lens", per stream tensors on the GPU, "sample": some tokens}.
    streams: any of "int4" (values, scale), "residual" (rvalues, rscale: the
    int4 code of what the int4 stream leaves), "sign" (sign, mean), and
    "sign_residual" (rvalues, rscale of what sign * mean leaves)."""
    lens = _lengths(case, seed)
    offsets = np.zeros(len(lens) + 1, np.int64)
    np.cumsum(lens, out=offsets[1:])
    parts = {}
    source = None
    for x in _embedding_blocks(lens, case.get("dim", 128), seed):
        if source is None:
            source = x
        out = {}
        if "int4" in streams:
            out["values"], out["scale"] = _int4(x)
            if "residual" in streams:
                out["rvalues"], out["rscale"] = _int4(x - out["values"].float() * out["scale"][:, None])
        if "sign" in streams:
            mean = x.abs().double().mean(dim=1).float()
            sign = torch.where(x >= 0, 1, -1).to(torch.int8)
            out["sign"], out["mean"] = sign, mean
            if "sign_residual" in streams:
                out["rvalues"], out["rscale"] = _int4(x - sign.float() * mean[:, None])
        for k, v in out.items():
            parts.setdefault(k, []).append(v)
    c = {k: torch.cat(v) if len(v) > 1 else v[0] for k, v in parts.items()}
    c.update(offsets=offsets, lens=lens, source=source)
    return c


def _query(case, seed, c):
    """f32 [B, qt, dim] on the GPU: per batch row noisy tokens of one document."""
    rng = np.random.default_rng([int(seed), 29])
    g = _generator(seed, 2)
    rows = []
    for _ in range(case["batch"]):
        doc = int(rng.integers(0, min(case["docs"], 8192)))
        start, n = int(c["offsets"][doc]), int(c["lens"][doc])
        pick = torch.from_numpy(start + rng.integers(0, n, size=case["qt"])).to(DEV)
        rows.append(_unit(c["source"][pick] + 0.1 * torch.randn(case["qt"], c["source"].shape[1], generator=g, device=DEV)))
    return torch.stack(rows).contiguous()


def _weights(case, seed):
    rng = np.random.default_rng([int(seed), 31])
    return rng.uniform(0.5, 1.5, size=(case["batch"], case["qt"])).astype(np.float32)


def _options(case, seed):
    o = {"reducer": case["reducer"]}
    if case["reducer"] == "weighted_maxsim":
        o["query_weights"] = _weights(case, seed)
    if case["reducer"] == "smoothsim":
        o["temperature"] = 0.1
    return o


def _candidates(case, seed):
    rng = np.random.default_rng([int(seed), 37])
    return rng.choice(case["docs"], size=case["candidates"], replace=False).astype(np.int64)


def _int4_handle(c):
    h = CudaInt4PackedDocs(_nibbles(c["values"]).cpu().numpy(), c["offsets"], int(c["values"].shape[1]), 1.0)
    scale = c["scale"].cpu().numpy()
    h.set_token_scale_vector(scale)
    return h, scale


def _top_buffers(case):
    return (torch.empty(case["batch"], case["k"], device=DEV),
            torch.empty(case["batch"], case["k"], dtype=torch.int64, device=DEV))


_STREAMS = {"int8_search": ("int4",), "int8_scores": ("int4",), "fp32_search": ("int4",), "rerank": ("int4",),
            "residual_search": ("int4", "residual"), "binary_search": ("sign",), "hamming_search": ("sign",),
            "binres_search": ("sign", "sign_residual")}


def _pack_input(case, seed):
    g = _generator(seed, 1)
    x = _unit(torch.randn(case["tokens"], case["dim"], generator=g, device=DEV))
    # Documents of 64 to 192 tokens until the tokens are used up.
    lens = np.random.default_rng([int(seed), 17]).integers(64, 193, size=case["tokens"] // 64 + 1)
    ends = np.minimum(np.cumsum(lens), case["tokens"])
    return x, np.concatenate([[0], ends]).astype(np.int64)


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op == "pack":
        s["x"], s["offsets"] = _pack_input(case, seed)
        return s
    c = _corpus(case, seed, _STREAMS[op])
    q = _query(case, seed, c)
    if op in ("int8_search", "int8_scores", "fp32_search", "rerank", "residual_search"):
        h, scale = _int4_handle(c)
        if op == "residual_search":
            h.set_residual_int4(_nibbles(c["rvalues"]).cpu().numpy(), 1.0, c["rscale"].cpu().numpy())
        s["handle"] = h
        s["packed"] = Int4PackedDocs(data=h, values=None, doc_offsets=c["offsets"], dim=int(q.shape[2]),
                                     num_docs=case["docs"], scale=1.0, device="cuda", token_scale=scale)
    else:
        # The sign of a zero embedding is +1, so +-1 values pack to the same bits.
        h = CudaPackedDocs(_sign_bits(c["sign"]).cpu().numpy(), c["offsets"], 128)
        scale = None
        if op == "binres_search" or case.get("token_scale"):
            scale = c["mean"].cpu().numpy()
            h.set_token_scale_vector(scale)
        if op == "binres_search":
            h.set_residual_int4(_nibbles(c["rvalues"]).cpu().numpy(), 1.0, c["rscale"].cpu().numpy())
        s["handle"] = h
        s["packed"] = PackedDocs(data=h, doc_offsets=c["offsets"], dim=128, num_docs=case["docs"], scale=None,
                                 device="cuda", token_scale=scale)
    if op in ("fp32_search", "rerank", "residual_search"):
        s["options"] = _options(case, seed)
    if op == "rerank":
        s["candidates"] = _candidates(case, seed)
    if op == "hamming_search":
        s["query"] = _sign_bits(q.view(-1, 128)).view(case["batch"], case["qt"], 16).contiguous()
    else:
        on_device = op in ("int8_scores", "binres_search") or (op == "int8_search" and not case["host"])
        s["query"] = q if on_device else q.cpu().numpy()
    if op == "int8_scores":
        s["out"] = torch.empty(case["batch"], case["docs"], device=DEV)
    elif op in ("hamming_search", "binres_search") or (op == "int8_search" and not case["host"]):
        s["top"] = _top_buffers(case)
    torch.cuda.synchronize()
    return s


# ----------------------------------------------------------------- one pass


def run(s):
    case, op = s["case"], s["case"]["op"]
    if op == "int8_search":
        if case["host"]:
            return topk_int4_maxsim(s["query"], s["packed"], case["k"], prefer_int8_query=True)
        s["handle"].topk_int8q_async(s["query"], case["k"], *s["top"])
        return s["top"]
    if op == "int8_scores":
        s["handle"].maxsim_int8q_async(s["query"], s["out"])
        return s["out"]
    if op == "fp32_search":
        return topk_int4_maxsim(s["query"], s["packed"], case["k"], **s["options"])
    if op == "rerank":
        return int4_maxsim(s["query"], s["packed"], candidate_indices=s["candidates"], **s["options"])
    if op == "residual_search":
        o = s["options"]
        args = (o["reducer"], o.get("query_weights"), o.get("temperature", 1.0))
        if case["candidates"]:
            return s["handle"].cascade_topk(s["query"], case["k"], case["candidates"], *args)
        return s["handle"].topk_score_batch(s["query"], case["k"], *args, residual=True)
    if op == "binary_search":
        return topk_maxsim(s["query"], s["packed"], case["k"])
    if op == "hamming_search":
        s["handle"].topk_hamming_async(s["query"], case["k"], *s["top"])
        return s["top"]
    if op == "binres_search":
        s["handle"].cascade_topk_async(s["query"], case["k"], case["candidates"], *s["top"])
        return s["top"]
    packed = pack_int4_symmetric_device(s["x"], s["offsets"], scale_granularity="token", values=False)
    return packed.data, packed.token_scale


# ------------------------------------------------------------- its least work


def work(case):
    op = case["op"]
    if op == "pack":
        # fp32 embeddings in, codes and one scale per token out; a maximum and
        # a scaled rounding per value.
        t, d = case["tokens"], case["dim"]
        return {"bytes": t * (4 * d + d // 2 + 4), "flops": 3 * t * d}
    mean = (case["lo"] + case["hi"]) / 2
    dim = case.get("dim", 128)
    rows = case["batch"] * case["qt"]
    tokens = case["docs"] * mean
    offsets = 8 * (case["docs"] + 1)
    query = rows * (dim // 8 if op == "hamming_search" else 4 * dim)
    top = 12 * case["batch"] * case.get("k", 0)
    int4 = dim // 2 + 4
    full = 2.0 * rows * tokens * dim
    if op == "int8_scores":
        return {"bytes": tokens * int4 + offsets + query + 4 * case["batch"] * case["docs"], "flops": full}
    if op == "rerank":
        t = case["candidates"] * mean
        return {"bytes": t * int4 + 16 * case["candidates"] + query + 4 * case["batch"] * case["candidates"],
                "flops": 2.0 * rows * t * dim}
    if op in ("int8_search", "fp32_search"):
        return {"bytes": tokens * int4 + offsets + query + top, "flops": full}
    if op == "residual_search":
        if case["candidates"]:
            cand = min(tokens, case["batch"] * case["candidates"] * mean)
            return {"bytes": tokens * int4 + cand * int4 + offsets + query + top,
                    "flops": full + 4.0 * case["qt"] * case["batch"] * case["candidates"] * mean * dim}
        return {"bytes": 2 * tokens * int4 + offsets + query + top, "flops": 2 * full}
    sign = dim // 8
    if op == "binres_search":
        cand = min(tokens, case["batch"] * case["candidates"] * mean)
        return {"bytes": tokens * (sign + 4) + cand * int4 + offsets + query + top,
                "flops": full + 4.0 * case["qt"] * case["batch"] * case["candidates"] * mean * dim}
    return {"bytes": tokens * (sign + (4 if case.get("token_scale") else 0)) + offsets + query + top, "flops": full}


def tolerance(case):
    # Integer dot products, Hamming scores, codes and the int8-query scan's
    # float64 sums: the same bits from any correct implementation.
    if case["op"] in ("int8_search", "int8_scores", "hamming_search", "pack"):
        return "exact"
    # fp32 similarities, their maxima and sums over the query tokens in 32
    # bits: 0.7e-7 to 2e-7 against exact() measured, the log-sum-exp's own
    # rounding more.
    if case.get("reducer") == "smoothsim":
        return {"rel": 4e-6, "max": 2e-5, "differ": 0.0}
    return {"rel": 1e-6, "max": 4e-6, "differ": 0.0}


# ---------------------------------------------------------- the same in 64 bits


def _reduce(sim, lens, reducer, tau):
    """sim f64 [T, R] of consecutive documents -> [docs, R]."""
    n, width = len(lens), int(lens.max())
    starts = np.concatenate([[0], np.cumsum(lens)[:-1]])
    idx = torch.from_numpy(starts[:, None] + np.minimum(np.arange(width)[None], lens[:, None] - 1)).to(sim.device)
    ok = torch.from_numpy(np.arange(width)[None] < lens[:, None]).to(sim.device)
    x = sim[idx.view(-1)].view(n, width, -1).masked_fill_(~ok[:, :, None], float("-inf"))
    if reducer in ("maxsim", "weighted_maxsim"):
        return x.amax(dim=1)
    if reducer == "smoothsim":
        return tau * torch.logsumexp(x / tau, dim=1)
    k = min(2 if reducer == "topk2" else 4, width)
    best = x.topk(k, dim=1).values
    kept = torch.from_numpy(np.minimum(lens, k)).to(sim.device)
    best = torch.where(torch.isfinite(best), best, torch.zeros_like(best))
    return best.sum(dim=1) / kept[:, None]


def _scores(sim_of, c, rows, batch, reducer="maxsim", tau=1.0, weights=None, row_factor=None):
    """f64 [batch, docs]; sim_of(a, b): similarities [b - a, rows] of tokens a .. b."""
    out = torch.empty(batch, len(c["lens"]), dtype=torch.float64, device=DEV)
    block = max(1, int(60_000_000 // (rows * int(c["lens"].max()))))
    for d in range(0, len(c["lens"]), block):
        e = min(d + block, len(c["lens"]))
        v = _reduce(sim_of(int(c["offsets"][d]), int(c["offsets"][e])), c["lens"][d:e], reducer, tau)
        if row_factor is not None:
            v = v * row_factor
        if weights is not None:
            v = v * weights
        out[:, d:e] = v.view(e - d, batch, -1).sum(dim=2).T
    return out


def _top(scores, k):
    """(score desc, id asc)."""
    order = torch.sort(scores, dim=1, descending=True, stable=True).indices[:, :k]
    return scores.gather(1, order), order


def _int8_query(q):
    """Query rows as the int8 path defines them: codes and their f32 step."""
    s = q.abs().amax(dim=-1) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(q / s[:, None]), -127, 127).double(), s.double()


def exact(case, seed):
    op = case["op"]
    if op == "pack":
        x, _ = _pack_input(case, seed)
        v, s = _int4(x)
        return _nibbles(v), s.double()
    c = _corpus(case, seed, _STREAMS[op])
    q = _query(case, seed, c).view(case["batch"] * case["qt"], -1)
    b, rows = case["batch"], q.shape[0]

    def part(values, scale, query):
        return lambda s, e: (values[s:e].double() @ query.T) * scale[s:e].double()[:, None]

    if op in ("int8_search", "int8_scores"):
        q8, sigma = _int8_query(q)
        f = _scores(part(c["values"], c["scale"], q8), c, rows, b, row_factor=sigma)
        return f if op == "int8_scores" else _top(f, case["k"])
    if op == "hamming_search":
        signs = torch.where(q >= 0, 1.0, -1.0).double()
        return _top(_scores(lambda s, e: c["sign"][s:e].double() @ signs.T, c, rows, b), case["k"])
    if op == "binary_search":
        if case["token_scale"]:
            sim = part(c["sign"], c["mean"], q.double())
        else:
            sim = lambda s, e: c["sign"][s:e].double() @ q.double().T  # noqa: E731
        return _top(_scores(sim, c, rows, b), case["k"])
    if op == "binres_search":
        q8, sigma = _int8_query(q)
        coarse_sim, res_sim = part(c["sign"], c["mean"], q8), part(c["rvalues"], c["rscale"], q8)
        coarse = _scores(coarse_sim, c, rows, b, row_factor=sigma)
        fine = _scores(lambda s, e: coarse_sim(s, e) + res_sim(s, e), c, rows, b, row_factor=sigma)
        return _top(_among(fine, coarse, case["candidates"]), case["k"])
    o = _options(case, seed)
    args = dict(reducer=o["reducer"], tau=o.get("temperature", 1.0))
    if "query_weights" in o:
        args["weights"] = torch.from_numpy(o["query_weights"]).to(DEV).double().view(-1)
    prefix = part(c["values"], c["scale"], q.double())
    if op == "fp32_search":
        return _top(_scores(prefix, c, rows, b, **args), case["k"])
    if op == "rerank":
        return _scores(prefix, c, rows, b, **args)[:, torch.from_numpy(_candidates(case, seed)).to(DEV)]
    residual = part(c["rvalues"], c["rscale"], q.double())
    fine = _scores(lambda s, e: prefix(s, e) + residual(s, e), c, rows, b, **args)
    if not case["candidates"]:
        return _top(fine, case["k"])
    coarse = _scores(prefix, c, rows, b, **args)
    return _top(_among(fine, coarse, case["candidates"]), case["k"])


def _among(fine, coarse, m):
    """Fine scores of each row's m best coarse documents, -inf elsewhere."""
    keep = _top(coarse, m)[1]
    out = torch.full_like(fine, float("-inf"))
    return out.scatter_(1, keep, fine.gather(1, keep))
