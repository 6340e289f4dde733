"""The work that users of this library have it do, as measurable cases.

A case is a dict of plain values: `op` names the entry point and the rest its
sizes and options.  `prepare` makes the inputs on the GPU (for the entry that
takes host arrays: in host memory), `run` makes one call, `work` counts what
the call cannot do without, `tolerance` says how far another correct
implementation may be off and `exact` gives the distances in 64 bits.

Sizes are those of bench.py's workloads (c1 to c5, ivf and their fp16 and
one-query forms) and generic ones between them.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

import mlxvs_amd

METRICS = ("l2", "inner_product", "cosine")


def listed():
    return [
        # the smallest call of the float path: a small collection, a small
        # batch (latency: launches and their gaps)
        dict(name="small_batch", op="dense", n=10_000, d=128, nq=100, k=10, metric="l2", f16=False,
             values="int"),
        # one interactive query against a million descriptors (HBM-bound)
        dict(name="one_query", op="dense", n=1_000_000, d=128, nq=1, k=10, metric="l2", f16=False,
             values="int"),
        # the headline use: ground truth / batch search over a million
        # SIFT-like descriptors (integers 0..255 held in float32)
        dict(name="descriptors", op="dense", n=1_000_000, d=128, nq=10_000, k=10, metric="l2",
             f16=False, values="int"),
        # the same size on learned (real-valued) features, with more
        # neighbours than a lane's list holds and ragged sizes throughout
        dict(name="features_ragged", op="dense", n=499_979, d=99, nq=2_741, k=50, metric="l2",
             f16=False, values="float"),
        # a batch search over a million large text embeddings in float32
        dict(name="embeddings", op="dense", n=1_000_000, d=1536, nq=10_000, k=10, metric="cosine",
             f16=False, values="float"),
        # the same embeddings held in half precision, inner product
        dict(name="embeddings_f16", op="dense", n=1_000_000, d=1536, nq=10_000, k=10,
             metric="inner_product", f16=True, values="float"),
        # a retrieval server's micro-batch over half a million sentence
        # embeddings (HBM-bound)
        dict(name="micro_batch", op="dense", n=500_000, d=768, nq=24, k=20, metric="inner_product",
             f16=False, values="float"),
        # search under a metadata filter (a bitset over the rows)
        dict(name="filtered", op="filtered", n=1_000_000, d=128, nq=1_000, k=10, metric="l2",
             f16=False, values="float", share=0.3),
        # the k-NN graph of a dataset in half precision (graph builders)
        dict(name="self_graph", op="self", n=200_000, d=256, k=64, metric="l2", f16=True),
        # binary codes: a million binarised embeddings, re-ranking depth 100
        dict(name="codes", op="hamming", n=1_000_000, nbytes=128, nq=10_000, k=100),
        # an inverted-file search (approximate index over the exact engine)
        dict(name="ivf", op="ivf", n=1_000_000, d=128, lists=1_024, probes=20, nq=10_000, k=10),
        # a distance outside the matrix products, on host arrays as a NumPy
        # program holds them
        dict(name="cityblock", op="pairwise", n=100_000, d=128, nq=1_000, k=10,
             distance="cityblock"),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    """One more case of the listed ones' ranges (sizes log-uniform, most of
    them odd; the work of a dense search at most that of `embeddings`)."""
    op = rng.choice(["dense"] * 6 + ["dense_f16"] * 2 + ["filtered", "self", "hamming", "ivf",
                                                          "pairwise"])
    k = _log(rng, 1, 100)
    if op in ("dense", "dense_f16", "filtered"):
        n = _log(rng, 10_000, 1_000_000)
        d = rng.choice([_log(rng, 16, 1536), rng.choice([32, 64, 96, 128, 256, 384, 768, 1024, 1536])])
        nq = _log(rng, 1, 10_000)
        case = dict(op="dense", n=n, d=d, nq=nq, k=k, metric=rng.choice(METRICS),
                    f16=op == "dense_f16",
                    values="float" if op == "dense_f16" or d > 256 else rng.choice(["int", "float"]))
        if op == "filtered":
            case.update(op="filtered", share=round(rng.uniform(0.05, 0.9), 3))
        return case
    if op == "self":
        return dict(op="self", n=_log(rng, 10_000, 200_000), d=_log(rng, 32, 256), k=min(k, 64),
                    metric=rng.choice(METRICS), f16=rng.choice([True, False]))
    if op == "hamming":
        return dict(op="hamming", n=_log(rng, 10_000, 1_000_000), nbytes=_log(rng, 16, 128),
                    nq=_log(rng, 1, 10_000), k=k)
    if op == "ivf":
        return dict(op="ivf", n=_log(rng, 100_000, 1_000_000), d=_log(rng, 32, 256),
                    lists=_log(rng, 128, 1_024), probes=_log(rng, 4, 32), nq=_log(rng, 1, 10_000),
                    k=min(k, 32))
    return dict(op="pairwise", n=_log(rng, 10_000, 100_000), d=_log(rng, 16, 128),
                nq=_log(rng, 10, 1_000), k=k,
                distance=rng.choice(["cityblock", "chebyshev", "canberra", "braycurtis"]))


# ---- inputs -------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rows(g, n: int, d: int, centres, values: str, f16: bool):
    """Mixture rows around `centres`: integers 0..255 (descriptors) or unit
    rows (embeddings), a block at a time."""
    out = torch.empty((n, d), device="cuda", dtype=torch.float16 if f16 else torch.float32)
    block = max(1, (1 << 26) // d)
    for lo in range(0, n, block):
        hi = min(n, lo + block)
        c = torch.randint(0, len(centres), (hi - lo,), generator=g, device="cuda")
        x = torch.randn((hi - lo, d), generator=g, device="cuda")
        if values == "int":
            x = (centres[c] + 20.0 * x).round_().clamp_(0.0, 255.0)
        else:
            x = torch.nn.functional.normalize(centres[c] + 0.7 * x)
        out[lo:hi] = x
    return out


def _centres(g, d: int, values: str, count: int):
    if values == "int":
        return torch.rand((count, d), generator=g, device="cuda") * 255.0
    return torch.randn((count, d), generator=g, device="cuda")


def prepare(case, seed):
    g = _gen(seed)
    op = case["op"]
    s = dict(case=case)
    if op in ("dense", "filtered"):
        cen = _centres(g, case["d"], case["values"], 1024 if case["d"] <= 256 else 256)
        s["base"] = _rows(g, case["n"], case["d"], cen, case["values"], case["f16"])
        s["queries"] = _rows(g, case["nq"], case["d"], cen, case["values"], case["f16"])
        if op == "filtered":
            words = (case["n"] + 31) // 32
            keep = torch.rand((words * 32,), generator=g, device="cuda") < case["share"]
            s["keep"] = keep[:case["n"]]
            bits = 1 << torch.arange(32, device="cuda", dtype=torch.int64)
            w = (keep.view(words, 32) * bits).sum(1)
            s["words"] = torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)
        nq = case["nq"]
    elif op == "self":
        cen = _centres(g, case["d"], "float", 512)
        s["base"] = _rows(g, case["n"], case["d"], cen, "float", case["f16"])
        nq = case["n"]
    elif op == "hamming":
        nb = case["nbytes"]
        s["base"] = torch.randint(0, 256, (case["n"], nb), generator=g, device="cuda",
                                  dtype=torch.uint8)
        # a query is a row of the base with about a twentieth of its bits flipped
        src = torch.randint(0, case["n"], (case["nq"],), generator=g, device="cuda")
        flip = torch.rand((case["nq"], nb, 8), generator=g, device="cuda") < 0.05
        bits = 1 << torch.arange(8, device="cuda")
        s["queries"] = s["base"][src] ^ (flip * bits).sum(2).to(torch.uint8)
        nq = case["nq"]
    elif op == "ivf":
        n, d, lists = case["n"], case["d"], case["lists"]
        cen = _centres(g, d, "int", lists).round_()
        x = _rows(g, n, d, cen, "int", False)
        s["queries"] = _rows(g, case["nq"], d, cen, "int", False)
        # the index as a program keeps it: rows grouped by their nearest centre
        half = cen.square().sum(1) * 0.5
        label = torch.empty((n,), device="cuda", dtype=torch.int64)
        block = 1 << 16
        for lo in range(0, n, block):
            label[lo:lo + block] = (x[lo:lo + block] @ cen.T - half).argmax(1)
        order = torch.argsort(label, stable=True)
        s["centers"], s["base"] = cen, x[order].contiguous()
        s["indices"] = order.to(torch.int32)
        s["offsets"] = torch.zeros((lists + 1,), device="cuda", dtype=torch.int32)
        s["offsets"][1:] = torch.bincount(label, minlength=lists).cumsum(0).to(torch.int32)
        nq = case["nq"]
    else:  # pairwise: non-negative features (histograms), in host memory
        r = np.random.default_rng(int(seed))
        s["base"] = r.gamma(2.0, 1.0, (case["n"], case["d"])).astype(np.float32)
        s["queries"] = r.gamma(2.0, 1.0, (case["nq"], case["d"])).astype(np.float32)
        return s
    s["ids"] = torch.empty((nq, case["k"]), device="cuda", dtype=torch.int32)
    s["dist"] = torch.empty((nq, case["k"]), device="cuda", dtype=torch.float32)
    s["stream"] = torch.cuda.current_stream().cuda_stream or None
    return s


# ---- one call ------------------------------------------------------------------


def run(state):
    c = state["case"]
    op = c["op"]
    if op == "pairwise":
        ids, dist = mlxvs_amd.pairwise_knn(state["base"], state["queries"], c["k"], c["distance"])
        return {"ids": ids, "dist": dist}
    base, ids, dist, st = state["base"], state["ids"], state["dist"], state["stream"]
    if op == "dense":
        q = state["queries"]
        mlxvs_amd.brute_force_knn_device(base.data_ptr(), c["n"], q.data_ptr(), c["nq"], c["d"],
                                         c["k"], c["metric"], ids.data_ptr(), dist.data_ptr(),
                                         f16=c["f16"], stream=st)
    elif op == "filtered":
        q = state["queries"]
        mlxvs_amd.brute_force_knn_filtered_device(
            base.data_ptr(), c["n"], q.data_ptr(), c["nq"], c["d"], c["k"], c["metric"],
            state["words"].data_ptr(), mlxvs_amd.FILTER_BITSET, ids.data_ptr(), dist.data_ptr(),
            f16=c["f16"], stream=st)
    elif op == "self":
        mlxvs_amd.knn_self_graph_device(base.data_ptr(), c["n"], c["d"], c["k"], c["metric"],
                                        ids.data_ptr(), dist.data_ptr(), f16=c["f16"], stream=st)
    elif op == "hamming":
        q = state["queries"]
        mlxvs_amd.hamming_knn_device(base.data_ptr(), c["n"], q.data_ptr(), c["nq"], c["nbytes"],
                                     c["k"], ids.data_ptr(), dist.data_ptr(), stream=st)
    else:
        q = state["queries"]
        mlxvs_amd.ivf_flat_search_device(
            state["centers"].data_ptr(), c["lists"], base.data_ptr(), c["n"],
            state["indices"].data_ptr(), state["offsets"].data_ptr(), c["d"], "l2", q.data_ptr(),
            c["nq"], c["k"], ids.data_ptr(), dist.data_ptr(), n_probes=c["probes"], stream=st)
    return {"ids": ids, "dist": dist}


def work(case):
    op, n, k = case["op"], case["n"], case["k"]
    if op == "hamming":
        nb, nq = case["nbytes"], case["nq"]
        return {"bytes": (n + nq) * nb + nq * k * 8, "flops": 2.0 * n * nq * nb * 8}
    d = case["d"]
    es = 2 if case.get("f16") else 4
    if op == "self":
        return {"bytes": n * d * es + n * k * 8, "flops": 2.0 * n * n * d}
    nq = case["nq"]
    if op == "ivf":
        cand = nq * case["probes"] * n / case["lists"]
        return {"bytes": min(n, cand) * d * 4 + (case["lists"] + nq) * d * 4 + nq * k * 8,
                "flops": 2.0 * d * (cand + nq * case["lists"])}
    if op == "pairwise":
        return {"bytes": (n + nq) * d * 4 + nq * k * 8, "flops": 2.0 * n * nq * d}
    share = case.get("share", 1.0)
    return {"bytes": n * d * es * share + nq * d * es + nq * k * 8, "flops": 2.0 * n * nq * d * share}


def tolerance(case):
    """Integer-valued rows have exact float32 sums under L2 and inner product,
    and Hamming distances are whole: every implementation agrees bit for bit
    (ties go to the lowest id).  Real-valued rows: float32 accumulation, and
    neighbours whose distances agree to that accuracy may change places (one
    exchange is 2 of the smallest float case's 480 ids)."""
    op = case["op"]
    if op == "hamming" or op == "ivf":
        return "exact"
    if op in ("dense", "filtered") and case["values"] == "int" and case["metric"] != "cosine":
        return "exact"
    return {"rel": 4e-6, "max": 2e-5, "differ": 0.01}


# ---- in 64 bits -----------------------------------------------------------------


def _best(score, k: int, nq: int, n: int, cells: int = 1 << 27):
    """The k largest of score(q0, q1, r0, r1) per query over all rows, in
    blocks (float64 [nq, k], largest first)."""
    qb = min(nq, 2048)
    rb = max(k, cells // qb)
    rows = []
    for q0 in range(0, nq, qb):
        best = None
        for r0 in range(0, n, rb):
            t = score(q0, min(nq, q0 + qb), r0, min(n, r0 + rb))
            t = torch.topk(t, min(k, t.shape[1]), dim=1).values
            best = t if best is None else torch.topk(torch.cat([best, t], 1), k, dim=1).values
        rows.append(best)
    return torch.cat(rows)


def exact(case, seed):
    s = prepare(case, seed)
    op, n, k = case["op"], case["n"], case["k"]
    if op == "ivf":
        return None  # whole numbers: compared bit for bit
    if op == "pairwise":
        if case["distance"] not in ("cityblock", "chebyshev"):
            return None
        b = torch.from_numpy(s["base"]).cuda().double()
        q = torch.from_numpy(s["queries"]).cuda().double()

        def score(q0, q1, r0, r1):
            t = (q[q0:q1, None] - b[None, r0:r1]).abs_()
            return -(t.sum(2) if case["distance"] == "cityblock" else t.amax(2))

        return {"ids": None, "dist": -_best(score, k, len(q), n, 1 << 20)}
    if op == "hamming":
        sh = torch.arange(8, device="cuda")

        def bits(x):
            return ((x.unsqueeze(-1) >> sh) & 1).reshape(len(x), -1).double()

        def score(q0, q1, r0, r1):
            q, b = bits(s["queries"][q0:q1]), bits(s["base"][r0:r1])
            return 2.0 * (q @ b.T) - b.sum(1) - q.sum(1, keepdim=True)

        return {"ids": None, "dist": -_best(score, k, case["nq"], n, 1 << 25)}
    metric = case["metric"]
    base = s["base"]
    queries = s["base"] if op == "self" else s["queries"]

    def score(q0, q1, r0, r1):
        q, b = queries[q0:q1].double(), base[r0:r1].double()
        if metric == "cosine":
            q = q / q.norm(dim=1, keepdim=True).clamp_min(1e-30)
            b = b / b.norm(dim=1, keepdim=True).clamp_min(1e-30)
        t = q @ b.T
        if metric == "l2":
            t = 2.0 * t - b.square().sum(1) - q.square().sum(1, keepdim=True)
        if op == "self":
            own = torch.arange(q0, q1, device="cuda")
            inside = (own >= r0) & (own < r1)
            t[torch.nonzero(inside).squeeze(1), own[inside] - r0] = -math.inf
        if op == "filtered":
            t[:, ~s["keep"][r0:r1]] = -math.inf
        return t

    best = _best(score, k, len(queries), n)
    return {"ids": None, "dist": (-best).clamp_min(0.0) if metric == "l2" else best}
