"""Workloads of the search, from its smallest call to its largest, for timing.

Every workload is what a program that uses the library does with one data set
(or one batch of data sets), through the public entry points of episdet.py:

  run      one complete search of a data set that is resident on the GPU,
           with the count tables built again inside the call (rebuild), as
           the benchmark's step does
  noalloc  the same answer through the entry point of serving loops, which
           allocates nothing on the device
  topk     the k best sets of a resident data set
  search   the reference-compatible call on host buffers: upload, search, free
  batch    many independent searches in one call
  tables   the contingency tables of explicit sets, as a program asks for
           after a search to report what it found

Genotypes are in Hardy-Weinberg proportions with minor-allele frequencies
uniform in [0.05, 0.5]; where "planted" is 1, one set of SNPs is associated
with the phenotype through a random penetrance table (0.1 baseline, 0.4
peak), else nothing is.  Classes are split by "case_pct".
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor-episdet_amd"))
import episdet  # noqa: E402

K2, MI = 0, 1
# C(n, order) * samples * 2^order * 2 of the most expensive listed search
LARGEST_FLOPS = 6.0e15


def _case(name, entry, order, score, snps, samples, case_pct=50, planted=1, **more):
    c = {"name": name, "entry": entry, "order": order, "score": score, "snps": snps, "samples": samples,
         "case_pct": case_pct, "planted": planted}
    c.update(more)
    return c


def listed():
    return [
        # The smallest pair search of the benchmark: one candidate-gene panel.
        _case("pairs_k2_512x2048", "run", 2, K2, 512, 2048, planted=0),
        # A pair scan of a filtered GWAS panel at an odd size.
        _case("pairs_k2_3001x9973", "run", 2, K2, 3001, 9973),
        # The benchmark's pair scan: uneven classes, mutual information.
        _case("pairs_mi_16384x65536", "run", 2, MI, 16384, 65536, case_pct=40),
        # A small triplet search asked for again and again by a server.
        _case("triplets_k2_200x1500_noalloc", "noalloc", 3, K2, 200, 1500),
        # An ordinary study: a few thousand samples, a thousand SNPs.
        _case("triplets_mi_1000x4000", "run", 3, MI, 1000, 4000),
        # A ragged size with uneven classes and no signal in the data.
        _case("triplets_k2_777x20001_30", "run", 3, K2, 777, 20001, case_pct=30, planted=0),
        # A biobank's sample axis: the published headline's samples, fewer SNPs.
        _case("triplets_k2_2048x262144", "run", 3, K2, 2048, 262144),
        # The 100 best triplets of a study, for a report or a replication list.
        _case("topk100_triplets_k2_1024x8192", "topk", 3, K2, 1024, 8192, k=100),
        # The reference's own call, host buffers in and answer out: pairs ...
        _case("search_pairs_k2_4096x65536", "search", 2, K2, 4096, 65536),
        # ... and triplets.
        _case("search_triplets_mi_400x10000", "search", 3, MI, 400, 10000),
        # Many uneven studies in one call (half of them 2-way, half K2).
        _case("batch_16x_700x20000", "batch", 0, 0, 700, 20000, jobs=16),
        # Tables of the triplets that a report lists.
        _case("tables_20000_triplets_2000x65536", "tables", 3, K2, 2000, 65536, sets=20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(["run", "run", "run", "noalloc", "topk", "search", "batch", "tables"])
    while True:
        order = rng.choice([2, 3])
        if order == 2:
            n, samples = _log_int(rng, 200, 16384), _log_int(rng, 1000, 262144)
        else:
            n, samples = _log_int(rng, 100, 4096), _log_int(rng, 1000, 262144)
        c = {"entry": entry, "order": order, "score": rng.choice([K2, MI]), "snps": n, "samples": samples,
             "case_pct": rng.choice([50, 50, 50, 40, 30, 20]), "planted": rng.choice([0, 1])}
        if entry == "topk":
            c["k"] = rng.choice([5, 20, 100, 500])
        elif entry == "batch":
            c.update(order=0, score=0, snps=min(n, 1000), samples=min(samples, 40000), jobs=rng.randrange(4, 25))
        elif entry == "tables":
            c["sets"] = _log_int(rng, 100, 40000)
        elif entry == "noalloc" and order == 3 and n > 1200:
            continue        # its scratch memory holds the tables of about 1400 SNPs
        if _flops(c) <= LARGEST_FLOPS and n * samples <= 16384 * 65536:
            return c


def _jobs(case):
    """(order, score, snps, samples) of every search of a case: a batch spreads
    its jobs from a third of its size to its size."""
    if case["entry"] != "batch":
        return [(case["order"], case["score"], case["snps"], case["samples"])]
    out = []
    for j in range(case["jobs"]):
        f = 1.0 / 3.0 + (2.0 / 3.0) * ((7 * j) % case["jobs"]) / max(1, case["jobs"] - 1)
        g = 1.0 / 3.0 + (2.0 / 3.0) * ((5 * j + 3) % case["jobs"]) / max(1, case["jobs"] - 1)
        out.append((2 + j % 2, (j // 2) % 2, max(8, int(case["snps"] * f)), max(64, int(case["samples"] * g))))
    return out


def _classes(case, samples):
    cases = max(1, samples * case["case_pct"] // 100)
    return cases, samples - cases


def _flops(case):
    if case["entry"] == "tables":
        return 2.0 * case["sets"] * case["samples"] * 2 ** case["order"]
    return sum(math.comb(n, o) * s * 2.0 * 2 ** o for o, _, n, s in _jobs(case))


def work(case):
    """Planes read once, answers written once; one multiply-add per sample for
    each of the 2^order independent cells of a set."""
    if case["entry"] == "tables":
        read = min(case["sets"] * case["order"], case["snps"]) * 2 * case["samples"] / 8
        return {"bytes": read + case["sets"] * 2 * 3 ** case["order"] * 4, "flops": _flops(case)}
    out = 16 * case.get("k", 1)
    return {"bytes": sum(n * 2 * s / 8 + out for _, _, n, s in _jobs(case)), "flops": _flops(case)}


# ------------------------------------------------------------------ inputs --

def _pack(g, words):
    """[rows, samples] genotypes -> [rows, 2, words] bit planes (sample s is bit
    31 - s % 32 of word s / 32) as int32 bit patterns."""
    rows, ns = g.shape
    shift = torch.arange(31, -1, -1, device=g.device, dtype=torch.int64)
    out = torch.zeros(rows, 2, words, dtype=torch.int32, device=g.device)
    for plane in range(2):
        bits = torch.zeros(rows, words * 32, dtype=torch.uint8, device=g.device)
        bits[:, :ns] = g == plane
        w = (bits.view(rows, words, 32).to(torch.int64) << shift).sum(-1)
        out[:, plane] = torch.where(w >= 2 ** 31, w - 2 ** 32, w).to(torch.int32)
    return out


def _genotypes(case, order, n, samples, seed):
    """Yields (class, first SNP, [rows, samples of the class] genotypes)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(seed)
    maf = 0.05 + 0.45 * torch.rand(n, generator=gen, device=dev)
    sets = {}
    if case["planted"]:
        snps = sorted(torch.randperm(n, generator=gen, device=dev)[:order].tolist())
        maf[snps] = 0.25 + 0.25 * torch.rand(order, generator=gen, device=dev)
        pen = 0.1 + 0.3 * (torch.rand(3 ** order, generator=gen, device=dev) < 0.25).to(torch.float32)
        hwe = torch.ones(1, device=dev)
        for s in snps:
            f = maf[s]
            hwe = (hwe[:, None] * torch.stack([(1 - f) ** 2, 2 * f * (1 - f), f * f])[None, :]).reshape(-1)
    for cls, ns in enumerate(_classes(case, samples)):
        if case["planted"]:
            cell = torch.multinomial(hwe * (pen if cls == 0 else 1 - pen), ns, replacement=True, generator=gen)
            for i, s in enumerate(snps):
                sets[s] = cell // 3 ** (order - 1 - i) % 3
        step = max(1, (1 << 27) // ns)
        for r0 in range(0, n, step):
            f = maf[r0:r0 + step, None]
            u = torch.rand(f.shape[0], ns, generator=gen, device=dev)
            g = (u >= (1 - f) ** 2).to(torch.uint8) + (u >= 1 - f * f).to(torch.uint8)
            for s in sets:
                if r0 <= s < r0 + f.shape[0]:
                    g[s - r0] = sets[s].to(torch.uint8)
            yield cls, r0, g


def _planes(case, order, n, samples, seed):
    """Host bit planes of both classes, padded to 1024 samples a row."""
    out = [np.zeros((n, 2, -(-ns // 1024) * 32), np.uint32) for ns in _classes(case, samples)]
    for cls, r0, g in _genotypes(case, order, n, samples, seed):
        out[cls][r0:r0 + g.shape[0]] = _pack(g, out[cls].shape[2]).cpu().numpy().view(np.uint32)
    return out


def _sets(case, seed):
    rng = np.random.default_rng(seed)
    s = np.sort(rng.integers(0, case["snps"] - case["order"] + 1, (case["sets"], case["order"])), axis=1)
    return (s + np.arange(case["order"])).astype(np.int32)       # strictly increasing


def prepare(case, seed):
    entry = case["entry"]
    state = {"case": case, "planes": [], "data": []}
    for j, (order, score, n, samples) in enumerate(_jobs(case)):
        planes = _planes(case, order, n, samples, seed * 1000 + j)
        nc, nt = _classes(case, samples)
        if entry == "search":
            state["planes"] = planes + [nc, nt]
        else:
            state["data"].append(episdet.Dataset(planes[0], planes[1], nc, nt))
    if entry == "batch":
        state["orders"] = [o for o, _, _, _ in _jobs(case)]
        state["scores"] = [s for _, s, _, _ in _jobs(case)]
    elif entry == "tables":
        state["sets"] = _sets(case, seed)
    if torch.cuda.is_available():
        torch.cuda.empty_cache()
    return state


def run(state):
    case = state["case"]
    entry, order, score = case["entry"], case["order"], case["score"]
    if entry == "search":
        packed, best, rounds, _ = episdet.search(order, score, *state["planes"])
        return {"set": list(episdet.unpack(order, packed)), "score": np.float32(best), "rounds": rounds}
    if entry == "batch":
        results, _ = episdet.run_batch(state["data"], state["orders"], state["scores"], rebuild=True)
        return {"set": np.array([r["idx"] for r in results]),
                "score": np.array([r["best_score"] for r in results])}
    data = state["data"][0]
    if entry == "tables":
        return data.tables(order, state["sets"])
    if entry == "topk":
        packed, scores, _ = data.topk(order, case["k"], score, rebuild=True)
        return {"sets": np.array([episdet.unpack(order, p) for p in packed]), "score": np.array(scores)}
    r = data.run(order, score, rebuild=True) if entry == "run" else data.run_noalloc(order, score)
    return {"set": list(r["idx"]), "score": r["best_score"]}


# ------------------------------------------------- the same in 64 bits -----

def _score_table(samples, score, dev):
    m = torch.arange(samples + 2, device=dev, dtype=torch.float64)
    if score == K2:
        return torch.lgamma(m + 1)
    p = m / samples
    return torch.where(p > 0, p * torch.log2(p.clamp_min(1e-300)), torch.zeros_like(p))


def _badness(counts, table, score, h_y):
    """Summed terms of the cells in the leading axis of counts = (cases, controls)."""
    a, b = (c.to(torch.int64) for c in counts)
    if score == K2:
        return (table[a + b + 1] - table[a] - table[b]).sum(0)
    return -(h_y + (table[a] + table[b] - table[a + b]).sum(0))


def _best(case, order, score, n, samples, seed, k):
    """The k best scores, ascending in badness, over every set."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    classes = _classes(case, samples)
    g = [torch.empty(n, ns, dtype=torch.uint8, device=dev) for ns in classes]
    for cls, r0, rows in _genotypes(case, order, n, samples, seed):
        g[cls][r0:r0 + rows.shape[0]] = rows
    table = _score_table(samples, score, dev)
    h_y = -sum(float(table[ns]) for ns in classes)
    best = torch.full((k,), math.inf, dtype=torch.float64, device=dev)

    def keep(bad):
        return torch.topk(torch.cat([best, bad]), k, largest=False).values

    if order == 2:
        hot = [torch.cat([(x == v) for v in range(3)]).to(torch.float32) for x in g]     # [3n, samples]
        step = max(1, (1 << 22) // n)
        for a0 in range(0, n, step):
            a1 = min(n, a0 + step)
            counts = []
            for h in hot:
                c = h.view(3, n, -1)[:, a0:a1].reshape(3 * (a1 - a0), -1) @ h.view(3, n, -1)[:, a0:].reshape(
                    3 * (n - a0), -1).T
                counts.append(c.view(3, a1 - a0, 3, n - a0).permute(0, 2, 1, 3).reshape(9, a1 - a0, n - a0))
            bad = _badness(counts, table, score, h_y)
            best = keep(bad[torch.ones_like(bad).triu(1).bool()])
        return best
    for x in range(n - 2):
        counts = [[], []]
        for cls, gc in enumerate(g):
            for gx in range(3):
                sub = gc[x + 1:, gc[x] == gx]                    # Y and Z among the samples of this X
                hot = torch.cat([(sub == v) for v in range(3)]).to(torch.float32)
                m = n - x - 1
                counts[cls].append((hot @ hot.T).view(3, m, 3, m).permute(0, 2, 1, 3).reshape(9, m, m))
        bad = _badness([torch.cat(c) for c in counts], table, score, h_y)
        best = keep(bad[torch.ones_like(bad).triu(1).bool()])
    return best


def exact(case, seed):
    """The scores of the best sets from one-hot products and log-gammas in 64
    bits (counts are whole numbers below 2^24, exact in float32 products); the
    sets themselves are whole numbers and have no such value."""
    entry, order, score = case["entry"], case["order"], case["score"]
    if entry == "tables":
        return None
    cost = sum(3.0 ** o * 2 * n ** o * s for o, _, n, s in _jobs(case))
    if cost > 1e15 or any(o == 3 and n > 1100 for o, _, n, _ in _jobs(case)):
        return None
    tops = [_best(case, o, s, n, ns, seed * 1000 + j, min(case.get("k", 1), math.comb(n, o))).cpu().numpy()
            for j, (o, s, n, ns) in enumerate(_jobs(case))]
    signed = [t if s == K2 else -t for t, (_, s, _, _) in zip(tops, _jobs(case))]
    if entry == "topk":
        return {"sets": None, "score": signed[0]}
    if entry == "batch":
        return {"set": None, "score": np.array([t[0] for t in signed])}
    if entry == "search":
        return {"set": None, "score": signed[0][0], "rounds": None}
    return {"set": None, "score": float(signed[0][0])}
