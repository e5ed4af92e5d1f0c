"""Workloads whose speed is measured: what a user of the library has it do, through its public entry points.

A training case is `sweeps` Gibbs sweeps of a corpus that is already loaded (a program loads once and sweeps
hundreds of times) and the topics read back; successive passes go on with the same chain.  An evaluation case is
the log-likelihood of a given state.  A serving case folds documents into a frozen model: a burst through the
server, one request alone through it, and one document on the plain path.

The documents come from the LDA generative process, drawn on the GPU: topics phi_k ~ Dir(0.01 V base) over a
Zipf(zipf) base distribution of the vocabulary, theta_d ~ Dir(0.1), at most 1024 topics.  The topic that each word
was drawn from is known, which gives the states that evaluation and serving start from the shape of a trained model.
"""
import math

import numpy as np
import torch

from lda_sc20_amd import ezlda


def listed():
    return [
        # A toy corpus, as in a test or a notebook: every sweep is a handful of launches over almost no data.
        dict(name="train_toy", kind="train", D=300, V=1000, K=20, dist="poisson", mean=60.0, zipf=0.0, head=-1.0,
             sweeps=50, graph=False, shortcut=True, evaluate=False, chunks=1),
        # The reference's CPU-sized job: 1M tokens, K = 64, 100 sweeps, replayed from a captured graph.
        dict(name="train_1m_k64", kind="train", D=10000, V=10000, K=64, dist="poisson", mean=100.0, zipf=0.0,
             head=-1.0, sweeps=100, graph=True, shortcut=True, evaluate=False, chunks=1),
        # Training with the perplexity watched after each sweep, on a mid-sized corpus with sizes that divide nothing.
        dict(name="train_watched_k300", kind="train", D=8011, V=5003, K=300, dist="lognormal", mean=211.0, zipf=1.0,
             head=-1.0, sweeps=10, graph=False, shortcut=True, evaluate=True, chunks=1),
        # The headline corpus (Zipf vocabulary, log-normal lengths, 1% of the words dense) at half its documents.
        dict(name="train_50m_k1024", kind="train", D=150000, V=102660, K=1024, dist="lognormal", mean=330.0,
             zipf=1.07, head=0.01, sweeps=20, graph=False, shortcut=True, evaluate=False, chunks=1),
        # Heavy-tailed lengths (Pareto, up to 20,000 tokens a document), K = 2048.
        dict(name="train_tailed_k2048", kind="train", D=40000, V=100000, K=2048, dist="pareto", mean=48.0, zipf=1.1,
             head=0.01, sweeps=10, graph=False, shortcut=True, evaluate=False, chunks=1),
        # Abstracts: many short documents, K = 4096, every word's counts dense.
        dict(name="train_short_k4096", kind="train", D=100000, V=20011, K=4096, dist="lognormal", mean=90.0, zipf=1.07,
             head=1.0, sweeps=10, graph=False, shortcut=True, evaluate=False, chunks=1),
        # The same kind of documents with K = 10000 topics (32-bit rows).
        dict(name="train_short_k10000", kind="train", D=50000, V=30000, K=10000, dist="lognormal", mean=90.0, zipf=1.07,
             head=-1.0, sweeps=10, graph=False, shortcut=True, evaluate=False, chunks=1),
        # Out of core: four chunks of documents streamed through the device each sweep.
        dict(name="train_chunked_k1024", kind="train", D=20000, V=20000, K=1024, dist="lognormal", mean=330.0,
             zipf=1.07, head=0.01, sweeps=10, graph=False, shortcut=True, evaluate=False, chunks=4),
        # Perplexity of a trained state.
        dict(name="evaluate_10m_k1024", kind="evaluate", D=30000, V=102660, K=1024, dist="lognormal", mean=330.0,
             zipf=1.07, head=0.01),
        # A burst of documents through the fold-in server: throughput with every slot taken.
        dict(name="serve_burst_k1024", kind="serve", D=10000, V=102660, K=1024, dist="lognormal", mean=300.0,
             zipf=1.07, head=0.01, requests=4096, slots=2048, sweeps=20),
        # One request alone in the server: latency at low load.
        dict(name="serve_one_k1024", kind="serve", D=10000, V=102660, K=1024, dist="lognormal", mean=300.0,
             zipf=1.07, head=0.01, requests=1, slots=2048, sweeps=20),
        # One document on the plain path (synchronous, no server thread).
        dict(name="fold_plain_k1024", kind="plain", D=10000, V=102660, K=1024, dist="lognormal", mean=300.0,
             zipf=1.07, head=0.01, requests=1, slots=64, sweeps=20),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["train"] * 7 + ["evaluate", "serve", "plain"])
    K = max(2, int(_log_uniform(rng, 16, 16383)))
    dist = rng.choice(["poisson", "lognormal", "lognormal", "pareto"])
    mean = round(_log_uniform(rng, 20, 60) if dist == "pareto" else _log_uniform(rng, 30, 600), 1)
    c = dict(kind=kind, V=int(_log_uniform(rng, 1000, 110000)), K=K, dist=dist, mean=mean,
             zipf=rng.choice([0.0, 1.0, 1.07, 1.1]))
    # V * K bounds the dense model of a case whose every word is dense, and the server's tables
    c["V"] = min(c["V"], 300000000 // K)
    c["head"] = rng.choice([-1.0, 0.01, 0.05, 1.0]) if c["V"] * K < 100000000 else rng.choice([-1.0, 0.01])
    tokens = _log_uniform(rng, 20000, 10000000)
    c["D"] = max(20, int(tokens / (mean * (5 if dist == "pareto" else 1))))
    if kind == "train":
        chunks = rng.choice([1, 1, 1, 1, 1, rng.randint(2, 6)])
        if chunks > 1:  # every word's counts are dense there
            c["V"] = min(c["V"], 100000000 // K)
        c.update(sweeps=rng.randint(5, 20), graph=chunks == 1 and rng.random() < 0.3, shortcut=rng.random() < 0.85,
                 evaluate=rng.random() < 0.2, chunks=chunks)
    elif kind == "evaluate":
        c["D"] = min(c["D"], int(4e9 / (c["K"] * mean * (5 if dist == "pareto" else 1))) + 20)
    else:
        c.update(requests=int(_log_uniform(rng, 1, 2000)) if kind == "serve" else 1,
                 slots=rng.choice([64, 500, 1024, 2048]), sweeps=20)
    return c


def _pick(weights, rows, gen):
    """One column of the integer `weights` for each of `rows`, with probability proportional to the weight."""
    n = weights.shape[1]
    cum = torch.cumsum(weights.reshape(-1), 0)
    end = cum[n - 1::n]
    first = torch.cat([end.new_zeros(1), end[:-1]])
    total = (end - first)[rows]
    u = (torch.rand(len(rows), generator=gen, device=rows.device, dtype=torch.float64) * total).long()
    at = torch.searchsorted(cum, first[rows] + torch.minimum(u, total - 1), right=True)
    return at - rows * n


def _weights(gamma):
    return (gamma / gamma.amax(1, keepdim=True).clamp_min(1e-30) * float(1 << 20)).long().clamp_min(0) + \
        (gamma.amax(1, keepdim=True) <= 0).long()


def _lengths(case, D, gen, dev):
    """Lengths of D documents: the quantiles of their distribution, shuffled, so that every seed has as many tokens."""
    mean = case["mean"]
    u = (torch.arange(D, dtype=torch.float64) + 0.5) / D
    x = math.sqrt(2.0) * torch.erfinv(2.0 * u - 1.0)  # quantiles of the normal law
    if case["dist"] == "poisson":
        n = torch.round(mean + math.sqrt(mean) * x)
    elif case["dist"] == "lognormal":  # sigma 0.8
        n = torch.exp(math.log(mean) - 0.32 + 0.8 * x)
    else:  # Pareto, shape 1.2, least length `mean`
        n = mean * (1.0 - u) ** (-1.0 / 1.2)
    return n.long().clamp(1, 20000).to(dev)[torch.randperm(D, generator=gen, device=dev)]


def _documents(case, seed, sizes):
    """(doc_off, words, topics) of sum(sizes) documents (each group of `sizes` with lengths of the whole
    distribution): the words, and the topics that they were drawn from, on the host."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 17)
    V, T, D = case["V"], min(case["K"], 1024), sum(sizes)
    n = torch.cat([_lengths(case, m, gen, dev) for m in sizes])
    base = torch.arange(1, V + 1, device=dev, dtype=torch.float64) ** -case["zipf"]
    conc = (0.01 * V * base / base.sum()).float()
    phi = _weights(torch._standard_gamma(conc.expand(T, V).contiguous(), generator=gen))
    ids = torch.randperm(V, generator=gen, device=dev)
    words, topics = [], []
    for d in range(0, D, 16384):
        m = n[d:d + 16384]
        theta = _weights(torch._standard_gamma(torch.full((len(m), T), 0.1, device=dev), generator=gen))
        k = _pick(theta, torch.repeat_interleave(torch.arange(len(m), device=dev), m), gen)
        words.append(ids[_pick(phi, k, gen)].int().cpu().numpy())
        topics.append(k.short().cpu().numpy().view(np.uint16))
    off = np.concatenate([[0], np.cumsum(n.cpu().numpy())]).astype(np.int64)
    return off, np.concatenate(words), np.concatenate(topics)


def _context(case, seed, **more):
    K, V = case["K"], case["V"]
    head = case["head"]
    return ezlda.Context(K=K, alpha=50.0 / K, beta=0.01, seed=2000 + seed,
                         dense_words=-1 if head < 0 else max(1, math.ceil(head * V)), **more)


def prepare(case, seed):
    if case["kind"] == "train":
        off, words, _ = _documents(case, seed, [case["D"]])
        ctx = _context(case, seed, shortcut=int(case["shortcut"]), num_chunks=case["chunks"])
        ctx.load(ezlda.Corpus(case["V"], off, words))
        return dict(case=case, ctx=ctx)
    if case["kind"] == "evaluate":
        off, words, z = _documents(case, seed, [case["D"]])
        ctx = _context(case, seed)
        ctx.load(ezlda.Corpus(case["V"], off, words), z0=z)
        return dict(case=case, ctx=ctx)
    # a frozen model of the first D documents; the others are the requests
    D, R = case["D"], case["requests"]
    off, words, z = _documents(case, seed, [D, R])
    ctx = _context(case, seed)
    ctx.load(ezlda.Corpus(case["V"], off[:D + 1], words[:off[D]]), z0=z[:off[D]])
    srv = ezlda.Server(ctx, max_slots=case["slots"], sweeps=case["sweeps"], hbm_budget_bytes=1 << 28, seed=seed + 7)
    return dict(case=case, srv=srv, ids=np.arange(R, dtype=np.uint32), off=off[D:] - off[D], words=words[off[D]:])


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        ctx, ll = state["ctx"], []
        if case["evaluate"]:
            for _ in range(case["sweeps"]):
                ctx.sweep(1)
                ll.append(ctx.loglik())
        elif case["graph"]:
            ctx.sweep_graph(case["sweeps"])
        else:
            ctx.sweep(case["sweeps"])
        z = ctx.get_topics()
        return dict(topics=z, loglik=np.array(ll)) if ll else dict(topics=z)
    if case["kind"] == "evaluate":
        return dict(loglik=np.float64(state["ctx"].loglik()))
    srv, ids, off, words = state["srv"], state["ids"], state["off"], state["words"]
    if case["kind"] == "plain":
        z, counts = srv.plain(0, words)
        return dict(topics=z, counts=counts)
    if len(ids) == 1:
        srv.submit(0, words)
    else:
        srv.submit_many(ids, off, words)
    done = [srv.wait(r) for r in ids.tolist()]
    return dict(topics=np.concatenate([x[0] for x in done]), counts=np.stack([x[1] for x in done]))


def _mean_length(case):
    """Expected tokens of a document."""
    if case["dist"] != "pareto":
        return case["mean"]
    # E[min(X, 20000)] of the Pareto law of shape 1.2 and scale m: m (1.2 - (m / 20000)^0.2) / 0.2
    m = case["mean"]
    return m * (1.2 - (m / 20000.0) ** 0.2) / 0.2


def work(case):
    """Per sweep each token's word is read (4 bytes), its topic read and written (2 + 2), and the sum over its
    document's topics formed (one multiply-add for each, about a third of min(n, K) of them)."""
    L, K = _mean_length(case), case["K"]
    terms = min(L, K) / 3.0
    if case["kind"] == "train":
        n = L * case["D"]
        one = 2 if case["evaluate"] else 1
        return {"bytes": n * case["sweeps"] * (8.0 + 6.0 * (one - 1)) + 2.0 * n,
                "flops": n * case["sweeps"] * 2.0 * terms * one}
    if case["kind"] == "evaluate":
        n = L * case["D"]
        return {"bytes": n * 6.0, "flops": n * 2.0 * terms}
    n = L * case["requests"]
    # words in once, topics and counts out once; the model's rows of the words, once
    return {"bytes": n * 6.0 + case["requests"] * K * 4.0 + min(n, case["V"]) * K * 4.0,
            "flops": n * case["sweeps"] * 2.0 * terms}


def exact(case, seed):
    """The log-likelihood of a given state, in 64 bits; topics are whole numbers and have no such value."""
    if case["kind"] != "evaluate":
        return None
    off, words, z = _documents(case, seed, [case["D"]])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    V, K, D = case["V"], case["K"], case["D"]
    beta = float(np.float32(0.01))
    alpha = float(np.float32(50.0 / K))
    w = torch.from_numpy(words).to(dev).long()
    t = torch.from_numpy(z.astype(np.int64)).to(dev)
    n = torch.from_numpy(np.diff(off)).to(dev)
    d = torch.repeat_interleave(torch.arange(D, device=dev), n)
    nk = torch.bincount(t, minlength=K).double()
    # distinct (document, topic) counts, in document order
    pair, cnt = torch.unique(d * K + t, return_counts=True)
    pd, pk, cnt = pair // K, pair % K, cnt.double()
    wt_pair, wt_cnt = torch.unique(w * K + t, return_counts=True)
    inv = 1.0 / (nk + V * beta)
    q = torch.zeros(V, dtype=torch.float64, device=dev).index_add_(
        0, wt_pair // K, wt_cnt.double() * inv[wt_pair % K]) + beta * inv.sum()
    first = torch.searchsorted(pd, torch.arange(D, device=dev))
    rows = torch.searchsorted(pd, torch.arange(D, device=dev), right=True) - first
    total = 0.0
    for a in range(0, len(w), 1 << 17):  # each token's sum over its document's topics
        ww, dd = w[a:a + (1 << 17)], d[a:a + (1 << 17)]
        m = rows[dd]
        tok = torch.repeat_interleave(torch.arange(len(ww), device=dev), m)
        j = torch.arange(len(tok), device=dev) - (torch.cumsum(m, 0) - m)[tok] + first[dd][tok]
        key = ww[tok] * K + pk[j]
        at = torch.searchsorted(wt_pair, key).clamp_max(len(wt_pair) - 1)
        nwk = torch.where(wt_pair[at] == key, wt_cnt[at], torch.zeros_like(at)).double()
        s = torch.zeros(len(ww), dtype=torch.float64, device=dev).index_add_(0, tok, cnt[j] * (nwk + beta) * inv[pk[j]])
        total += float(torch.log((s + alpha * q[ww]) / (n[dd].double() + K * alpha)).sum())
    return dict(loglik=np.float64(total))
