"""Performance cases of the search library: what a user's program has it do.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges. ``prepare`` makes the
inputs and the index that a program holds before the call, ``run`` is one call through the public
Python API, ``work`` the bytes and operations the call cannot do without, ``tolerance`` the
agreement asked of the outputs and ``exact`` the same outputs in 64-bit arithmetic by plain torch.

The kinds of call:
  flat    FlatIndex.search: exact top-k over all rows (or over an allowed-id filter).
  ivf     IvfPqIndex.search over probed lists, optionally re-ranked from stored vectors.
  add     IvfPqIndex.add into an empty trained index (cell assignment and PQ encoding).
  train   IvfPqIndex.train (coarse k-means and one k-means per PQ sub-space).

Row and query distributions follow quiver_amd/datasets.py: "int" is an integer-valued mixture in
0..255 (SIFT-like descriptors), "unit" an anisotropic mixture on the unit sphere (word or image
embeddings), "normal" N(0, 1).
"""

from __future__ import annotations

import math

import numpy as np
import torch

import quiver_amd as quiver

_DEVICE = "cuda"


# ---- the cases --------------------------------------------------------------------------------


def _flat(name, n, dim, nq, k, metric="l2", data="int", host=False, allowed=1.0):
    return dict(name=name, kind="flat", n=n, dim=dim, nq=nq, k=k, metric=metric, data=data, host=host,
                allowed=allowed)


def _ivf(name, n, dim, nq, k, nlist, m, nprobe, refine=0, metric="l2", data="int", host=False):
    return dict(name=name, kind="ivf", n=n, dim=dim, nq=nq, k=k, nlist=nlist, m=m, nprobe=nprobe, refine=refine,
                metric=metric, data=data, host=host)


def listed():
    return [
        # A small collection searched with a handful of questions at a time (README quick start,
        # the 10,000 x 128 configuration): launches and host work count.
        _flat("flat_small_100q", 10_000, 128, 100, 10, data="normal", host=True),
        # Online serving: one query against a million descriptors.
        _flat("flat_1m_1q", 1_000_000, 128, 1, 10, host=True),
        # Online serving with request batching, queries already on the GPU.
        _flat("flat_1m_32q", 1_000_000, 128, 32, 10),
        # A medium offline batch over embeddings with inner product: ragged sizes, a larger k.
        _flat("flat_ip_1003q", 300_007, 96, 1_003, 30, metric="ip", data="normal"),
        # The headline batch: 10,000 queries against 1,000,000 x 128, k = 10.
        _flat("flat_1m_10kq", 1_000_000, 128, 10_000, 10),
        # Cosine search restricted to an allowed tenth of the ids, through host arrays.
        _flat("flat_cosine_filter", 1_183_514, 100, 10_000, 10, metric="cosine", data="unit", host=True, allowed=0.1),
        # Text-embedding width (768): rows too wide for one register-resident query block.
        _flat("flat_wide_768", 200_003, 768, 2_000, 10, data="normal"),
        # IVF-PQ serving: one query, 32 probes.
        _ivf("ivf_1m_1q", 1_000_000, 128, 1, 10, 2048, 32, 32, host=True),
        # The headline IVF-PQ batch: nlist 2048, m 32, nprobe 32.
        _ivf("ivf_1m_10kq", 1_000_000, 128, 10_000, 10, 2048, 32, 32),
        # Cosine IVF-PQ with exact re-ranking of 8 k candidates from stored vectors.
        _ivf("ivf_cosine_refine", 1_183_514, 100, 10_000, 10, 2048, 25, 16, refine=8, metric="cosine", data="unit"),
        # Building an index: a batch of vectors assigned and encoded into an empty trained index.
        dict(name="ivf_add", kind="add", n=200_000, dim=128, nlist=2048, m=32, metric="l2", data="int"),
        # Training on a sample.
        dict(name="ivf_train", kind="train", n=50_000, dim=64, nlist=512, m=16, metric="l2", data="normal"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["flat", "ivf", "add"], [6, 4, 1])[0]
    metric = rng.choice(["l2", "l2", "ip", "cosine"])
    data = "unit" if metric == "cosine" else rng.choice(["int", "normal"])
    if kind == "flat":
        wide = rng.random() < 0.25
        dim = _log_int(rng, 129, 1024) if wide else rng.randint(16, 128)
        n = _log_int(rng, 5_000, 200_000 if wide else 1_000_000)
        # At most 1e12 operations a call: the largest listed batch takes 2.6e12.
        nq = _log_int(rng, 1, max(2, min(10_000, int(1e12 / (2.0 * n * dim)))))
        k = rng.choice([1, 10, 10, 10, 20, 50, 100])
        allowed = rng.choice([1.0, 1.0, 1.0, 0.5, 0.1, 0.01])
        case = _flat("", n, dim, nq, k, metric, data, rng.random() < 0.4, allowed)
    else:
        m, dsub = rng.choice([8, 16, 25, 32, 48]), rng.choice([2, 3, 4, 4, 8])
        n = _log_int(rng, 20_000, 1_000_000)
        nlist = _log_int(rng, 64, min(2048, n // 64))
        if kind == "add":
            n = min(n, 200_000)
            case = dict(name="", kind="add", n=n, dim=m * dsub, nlist=nlist, m=m, metric=metric, data=data)
        else:
            # At most 6e9 bytes of codes scanned a call: the largest listed batch reads 5e9.
            nprobe = _log_int(rng, 1, 64)
            nq = _log_int(rng, 1, max(2, min(10_000, int(6e9 / (n * m * min(1.0, nprobe / nlist))))))
            k = rng.choice([1, 10, 10, 10, 50, 100])
            refine = rng.choice([0, 0, 4]) if k <= 50 else 0
            case = _ivf("", n, m * dsub, nq, k, nlist, m, nprobe, refine, metric, data, rng.random() < 0.4)
    del case["name"]
    return case


# ---- inputs -----------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device=_DEVICE)
    g.manual_seed(seed)
    return g


def _vectors(case, seed, counts):
    """One float32 device matrix per entry of counts, all of the same mixture."""
    g, dim = _generator(seed), case["dim"]
    normal = lambda *shape: torch.randn(shape, generator=g, device=_DEVICE)  # noqa: E731
    uniform = lambda *shape: torch.rand(shape, generator=g, device=_DEVICE)  # noqa: E731
    if case["data"] == "normal":
        return [normal(n, dim) for n in counts]
    comps = 64 if case["data"] == "int" else 256
    if case["data"] == "int":
        means, sigma = 160.0 * uniform(comps, dim), 8.0 + 24.0 * uniform(comps, 1)
    else:
        means, sigma = normal(comps, dim), torch.exp(2.0 * uniform(1, dim) - 1.5).expand(comps, dim)
    out = []
    for n in counts:
        c = torch.randint(0, comps, (n,), generator=g, device=_DEVICE)
        x = torch.addcmul(means[c], sigma[c], normal(n, dim))
        out.append(x.round_().clamp_(0.0, 255.0) if case["data"] == "int" else torch.nn.functional.normalize(x))
    return out


def _allowed(case, seed):
    """The allowed ids (sorted), or None without a filter."""
    if case["allowed"] >= 1.0:
        return None
    count = max(1, int(round(case["n"] * case["allowed"])))
    return np.sort(torch.randperm(case["n"], generator=_generator(seed + 1), device=_DEVICE)[:count].cpu().numpy())


def _nearest(x, c):
    """Nearest rows of c (float64), in chunks."""
    c2 = (c * c).sum(1)
    return torch.cat([(c2 - 2.0 * (b @ c.T)).argmin(1) for b in x.split(32_768)])


def _means(x, cell, k, grid):
    """Per-cell means of x rounded to a grid: the sums are exact, so they do not depend on order."""
    x = torch.round(x * grid)
    s = torch.zeros(k, x.shape[1], dtype=torch.float64, device=x.device).index_add_(0, cell, x)
    cnt = torch.bincount(cell, minlength=k).clamp_(min=1).to(torch.float64)
    return s / (grid * cnt[:, None])


def _trained(case, x):
    """Coarse centroids and PQ codebook a few k-means steps from a sample of x (plain torch)."""
    nlist, m = case["nlist"], case["m"]
    grid = float(1 << 20)
    step = max(1, x.shape[0] // max(32_768, 16 * nlist))
    sample = x[::step].to(torch.float64)
    if case["metric"] == "cosine":
        sample = torch.nn.functional.normalize(sample)
    cent = sample[torch.linspace(0, sample.shape[0] - 1, nlist, device=x.device).long()]
    for _ in range(3):
        cell = _nearest(sample, cent)
        got = torch.bincount(cell, minlength=nlist) > 0
        cent = torch.where(got[:, None], _means(sample, cell, nlist, grid), cent)
    if case["metric"] == "cosine":
        cent = torch.nn.functional.normalize(cent)
    cent = cent.to(torch.float32)
    res = (sample - cent.to(torch.float64)[_nearest(sample, cent.to(torch.float64))])[:16_384]
    books = []
    for sub in res.split(case["dim"] // m, dim=1):
        book = sub[torch.linspace(0, sub.shape[0] - 1, 256, device=x.device).long()]
        for _ in range(2):
            cell = _nearest(sub, book)
            got = torch.bincount(cell, minlength=256) > 0
            book = torch.where(got[:, None], _means(sub, cell, 256, grid), book)
        books.append(book.to(torch.float32))
    return cent, torch.stack(books)


def _empty_ivf(case):
    return quiver.IvfPqIndex(case["dim"], case["metric"], nlist=case["nlist"], m=case["m"],
                             store_vectors=case.get("refine", 0) > 0)


def prepare(case, seed):
    if case["kind"] == "train":
        (x,) = _vectors(case, seed, [case["n"]])
        return dict(case=case, x=x.cpu().numpy())
    if case["kind"] == "add":
        (x,) = _vectors(case, seed, [case["n"]])
        cent, book = _trained(case, x)
        return dict(case=case, x=x.cpu().numpy(), centroids=cent.cpu().numpy(), codebook=book.cpu().numpy())
    x, q = _vectors(case, seed, [case["n"], case["nq"]])
    state = dict(case=case, queries=q.cpu().numpy() if case["host"] else q)
    if case["kind"] == "flat":
        index = quiver.FlatIndex(case["dim"], case["metric"])
        state["filter"] = _allowed(case, seed)
    else:
        index = _empty_ivf(case)
        cent, book = _trained(case, x)
        index.set_trained(cent.cpu().numpy(), book.cpu().numpy())
    index.add(x.cpu().numpy())
    state["index"] = index
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "flat":
        return state["index"].search(state["queries"], k=case["k"], filter=state["filter"])
    if case["kind"] == "ivf":
        return state["index"].search(state["queries"], k=case["k"], nprobe=case["nprobe"],
                                     refine_factor=case["refine"])
    index = _empty_ivf(case)
    if case["kind"] == "add":
        index.set_trained(state["centroids"], state["codebook"])
        index.add(state["x"])
        return index.lists()
    index.train(state["x"])
    return index.centroids, index.codebook


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    n, dim = float(case["n"]), case["dim"]
    if case["kind"] == "flat":
        rows, nq = n * case["allowed"], case["nq"]
        return {"bytes": 4.0 * dim * (rows + nq) + 12.0 * nq * case["k"], "flops": 2.0 * rows * dim * nq}
    nlist, m = case["nlist"], case["m"]
    trained = 4.0 * dim * (nlist + 256)
    if case["kind"] == "ivf":
        # Coarse scores, one table of m x 256 entries a query, one addition per sub-space of every
        # probed code, and with refine the exact distance of each kept candidate.
        nq, probed = case["nq"], n * min(1.0, case["nprobe"] / nlist)
        keep = case["k"] * case["refine"]
        codes = min(n, nq * probed) * m
        return {"bytes": codes + trained + 4.0 * dim * (nq + min(n, nq * keep)) + 12.0 * nq * case["k"],
                "flops": nq * (2.0 * nlist * dim + 2.0 * 256 * dim + probed * m + 2.0 * keep * dim)}
    if case["kind"] == "add":
        return {"bytes": 4.0 * dim * n + trained + n * (m + 8.0), "flops": n * (2.0 * nlist * dim + 2.0 * 256 * dim)}
    # 20 iterations of the coarse k-means and of the sub-space ones.
    return {"bytes": 4.0 * dim * n + trained, "flops": 20.0 * n * (2.0 * nlist * dim + 2.0 * 256 * dim)}


def tolerance(case):
    # Distances, codes and trained state are promised bit for bit (the arithmetic order of every
    # sum is part of the interface, and equal distances come in order of row), so nothing may differ.
    return "exact"


# ---- 64-bit results ---------------------------------------------------------------------------


def _distances(case, q, x):
    """float64 [nq, n] distances of the case's metric."""
    if case["metric"] == "l2":
        d = (q @ x.T).mul_(-2.0).add_((x * x).sum(1)).add_((q * q).sum(1)[:, None])
        return d.clamp_(min=0.0)
    return (q @ x.T).neg_().add_(1.0)


def exact(case, seed):
    """(None, distances): labels are positions, not numbers. None for add and train, whose outputs
    follow from comparisons (codes) or amplify rounding over iterations (k-means)."""
    if case["kind"] not in ("flat", "ivf"):
        return None
    n, nq, k = case["n"], case["nq"], case["k"]
    x32, q32 = _vectors(case, seed, [n, nq])
    x, q = x32.to(torch.float64), q32.to(torch.float64)
    if case["metric"] == "cosine":
        x, q = torch.nn.functional.normalize(x), torch.nn.functional.normalize(q)
    out = torch.full((nq, k), math.inf, dtype=torch.float64, device=_DEVICE)
    chunk = max(1, int(1.5e8 / n))
    if case["kind"] == "flat":
        allowed = _allowed(case, seed)
        if allowed is not None:
            x = x[torch.from_numpy(allowed).to(_DEVICE)]
        take = min(k, x.shape[0])
        for b in range(0, nq, chunk):
            d = _distances(case, q[b:b + chunk], x)
            out[b:b + chunk, :take] = d.topk(take, dim=1, largest=False).values
    else:
        cent, book = (t.to(torch.float64) for t in _trained(case, x32))
        if case["metric"] == "ip":
            cell = torch.cat([(b @ cent.T).argmax(1) for b in x.split(32_768)])
        else:
            cell = _nearest(x, cent)
        near = cent[cell]
        dsub = case["dim"] // case["m"]
        approx = torch.cat([near[:, j * dsub:(j + 1) * dsub] + book[j][_nearest(
            (x - near)[:, j * dsub:(j + 1) * dsub], book[j])] for j in range(case["m"])], dim=1)
        nprobe, refine = min(case["nprobe"], case["nlist"]), case["refine"]
        keep = min(n, k * max(1, refine))
        for b in range(0, nq, chunk):
            qb = q[b:b + chunk]
            probes = _distances(case, qb, cent).topk(nprobe, dim=1, largest=False).indices
            probed = torch.zeros(qb.shape[0], case["nlist"], dtype=torch.bool, device=_DEVICE).scatter_(1, probes, True)
            d = _distances(case, qb, approx).masked_fill_(~probed[:, cell], math.inf)
            best = d.topk(keep, dim=1, largest=False)
            d = best.values
            if refine:
                rows = x[best.indices]
                full = ((qb[:, None] - rows) ** 2).sum(2) if case["metric"] == "l2" else \
                    1.0 - (rows * qb[:, None]).sum(2)
                d = full.masked_fill_(torch.isinf(d), math.inf)
            take = min(k, keep)
            out[b:b + chunk, :take] = d.topk(take, dim=1, largest=False).values
    out = out.to(_DEVICE)
    return None, out.cpu().numpy() if case["host"] else out
