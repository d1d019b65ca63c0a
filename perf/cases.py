"""Performance cases: the work a user of sparkx_amd has it do, through its public entry points.

Every case is a dict of plain values.  `prepare` builds what a user's program holds before
the call (graphs come from torch on the GPU, seeded; the same families as bench.py: R-MAT
with a, b, c = .57, .19, .19, Erdos-Renyi, canonical k-mer graphs of a mutated genome, the
de Bruijn graphs of the reference's accuracy fixtures), `run` is one pass through the
public API with its results in host arrays, as the API returns them, `exact` is the same
result in 64-bit torch where it has a value outside this repository, and `work` is the
traffic one pass cannot do without.

Kinds:
  new       HyperBall(g, p) from a host CSR and one centrality: create, stage, run, read
  hyperball run() of a staged graph, then centralities or accumulators
  batch     HyperBallBatch.run() over many graphs of mixed size and precision, then every
            graph's accumulators
  exact     exact BFS centrality of a source range, from a host CSR
  ingest    MatrixMarket text to CSR (read_mtx)
  walks     anytime ranking of a staged graph from walk counts (Surrogate.rank_walks)
  gradient  forward and backward of the surrogate network over a training set
"""
import math
import random

import numpy as np
import torch

from sparkx_amd import Graph, HyperBall
from sparkx_amd.batch import HyperBallBatch
from sparkx_amd.exact import ExactClosenessCentrality, ExactHarmonicCentrality
from sparkx_amd.ingest import read_mtx
from sparkx_amd.surrogate import N_PARAMS, Surrogate

DEV = "cuda"


def listed():
    return [
        # the smallest call: a graph of a few thousand nodes, once through, end to end
        dict(name="new-er-4k-p6", kind="new", graph="er", n=4096, samples=32768, p=6, out="closeness"),
        # the Erdos-Renyi configuration (n = 65,536, m = 2^20, p = 6): launches and latency
        dict(name="run-er-64k-p6", kind="hyperball", graph="er", n=65536, samples=1 << 20, p=6, iters=0,
             out="accumulators"),
        # a mid-size social-like graph at the library's default precision, every centrality read
        dict(name="run-rmat-20-p8", kind="hyperball", graph="rmat", scale=20, factor=16, p=8, iters=0, out="all"),
        # the headline configuration: R-MAT-24, p = 7, to convergence, one centrality read
        dict(name="run-rmat-24-p7", kind="hyperball", graph="rmat", scale=24, factor=16, p=7, iters=0,
             out="closeness"),
        # the genome configuration: long low-degree chains, 64 iterations
        dict(name="run-kmer-4m-p6", kind="hyperball", graph="kmer", genome=4_000_000, copies=8, k=21, p=6, iters=64,
             out="harmonic"),
        # the accuracy profile's graph (DNA de Bruijn, k = 7) at a high precision
        dict(name="run-dbg-16k-p12", kind="hyperball", graph="dbg", sigma=4, k=7, p=12, iters=0, out="closeness"),
        # many graphs of mixed size and precision together
        dict(name="batch-32", kind="batch", count=32, lo=12, hi=18, sizes=1),
        # ground truth of the accuracy profile: every node's exact closeness
        dict(name="exact-dbg-16k-all", kind="exact", graph="dbg", sigma=4, k=7, sources=16384, out="closeness"),
        # ground truth on a sample of a larger graph
        dict(name="exact-rmat-20-2048", kind="exact", graph="rmat", scale=20, factor=16, sources=2048,
             out="harmonic"),
        # a MatrixMarket file read into a CSR
        dict(name="ingest-rmat-20", kind="ingest", graph="rmat", scale=20, factor=16),
        # an anytime ranking of a staged graph
        dict(name="walks-rmat-22", kind="walks", graph="rmat", scale=22, factor=16, passes=2),
        # a training step's gradient of the surrogate over a graph's nodes
        dict(name="gradient-1m", kind="gradient", count=1_000_003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["new", "hyperball", "hyperball", "hyperball", "batch", "exact", "ingest", "walks", "gradient"])
    if kind == "gradient":
        return dict(kind=kind, count=_log(rng, 3_001, 4_000_000) | 1)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 32), lo=12, hi=rng.randint(14, 18), sizes=rng.randrange(1 << 20))
    if kind == "new":
        n = _log(rng, 1000, 100_000)
        return dict(kind=kind, graph="er", n=n, samples=int(n * rng.uniform(2, 16)), p=rng.randint(4, 10),
                    out=rng.choice(["closeness", "harmonic", "lin"]))
    family = rng.choice(["er", "rmat", "dbg"] if kind == "exact" else ["rmat", "er"] if kind in ("ingest", "walks")
                        else ["er", "rmat", "rmat", "kmer", "dbg"])
    top = dict(hyperball=2_000_000, exact=200_000, ingest=500_000, walks=2_000_000)[kind]
    if family == "er":
        n = _log(rng, 4_001, top) | 1
        c = dict(kind=kind, graph="er", n=n, samples=int(n * rng.uniform(2, 16)))
    elif family == "rmat":
        c = dict(kind=kind, graph="rmat", scale=rng.randint(13, int(math.log2(top)) + 1), factor=rng.randint(4, 16))
        n = 1 << c["scale"]
    elif family == "kmer":
        c = dict(kind=kind, graph="kmer", genome=_log(rng, 100_000, 4_000_000), copies=rng.randint(2, 8),
                 k=rng.choice([17, 21, 25, 31]))
        n = 2 * c["genome"]
    else:
        sigma, k = rng.choice([(4, 6), (4, 7), (4, 8), (20, 3), (3, 9)])
        c = dict(kind=kind, graph="dbg", sigma=sigma, k=k)
        n = sigma**k
    if kind == "hyperball":
        # registers of at most half a GiB: higher precisions for the smaller graphs
        c["p"] = rng.randint(4, max(4, min(13, int(math.log2(2.0**29 / n)))))
        c["iters"] = rng.choice([8, 32, 64]) if family == "kmer" else rng.choice([0, 0, 4])
        c["out"] = rng.choice(["closeness", "harmonic", "lin", "accumulators", "all"])
    elif kind == "exact":
        c["sources"] = min(n, _log(rng, 65, 4096))
        c["out"] = rng.choice(["closeness", "harmonic"])
    elif kind == "walks":
        c["passes"] = rng.choice([2, 3])
    return c


# ---- graphs ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


def _csr(n, u, v, simple=True):
    """Symmetric CSR of an edge list on the GPU, lists ascending; `simple` drops loops and
    repeated edges (a loop kept counts once)."""
    if simple:
        keep = u != v
        u, v = u[keep], v[keep]
    key = torch.cat([u * n + v, (v * n + u)[u != v]])
    del u, v
    key = torch.unique(key) if simple else torch.sort(key)[0]
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(torch.div(key, n, rounding_mode="floor"), minlength=n), 0)
    return off, key % n


def _rmat(scale, factor, gen):
    m = factor << scale
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        x = torch.rand(m, device=DEV, generator=gen)
        u = u * 2 + (x >= 0.76)
        v = v * 2 + (((x >= 0.57) & (x < 0.76)) | (x >= 0.95))
    return _csr(1 << scale, u, v)


def _er(n, samples, gen):
    return _csr(n, torch.randint(n, (samples,), device=DEV, generator=gen),
                torch.randint(n, (samples,), device=DEV, generator=gen))


def _kmer(genome, copies, k, gen):
    """Canonical k-mers of `copies` copies of a random genome with 0.5% substitutions;
    consecutive k-mers of a copy are neighbours.  The last ids, up to a fixed number of
    nodes, are k-mers without a neighbour."""
    base = torch.randint(4, (genome,), device=DEV, generator=gen)
    mers = []
    for _ in range(copies):
        hit = torch.rand(genome, device=DEV, generator=gen) < 0.005
        seq = torch.where(hit, (base + torch.randint(1, 4, (genome,), device=DEV, generator=gen)) % 4, base)
        w = genome - k + 1
        fwd = torch.zeros(w, dtype=torch.int64, device=DEV)
        rev = torch.zeros(w, dtype=torch.int64, device=DEV)
        for i in range(k):
            fwd = fwd * 4 + seq[i:i + w]
            rev = rev * 4 + (3 - seq[k - 1 - i:k - 1 - i + w])
        mers.append(torch.minimum(fwd, rev))
    ids, inv = torch.unique(torch.cat(mers), return_inverse=True)
    inv = inv.reshape(copies, -1)
    n = _kmer_nodes(genome, copies, k)
    assert ids.numel() <= n
    return _csr(n, inv[:, :-1].reshape(-1), inv[:, 1:].reshape(-1))


def _kmer_nodes(genome, copies, k):
    return int(genome * (1 + 1.1 * copies * (1 - 0.995**k))) + 4000


def _dbg(sigma, k, gen):
    """De Bruijn graph of all words of length k (arcs w -> w's last k - 1 letters and one
    more, both ways, repeats and loops kept), its nodes renumbered by the seed."""
    n = sigma**k
    u = torch.arange(n, device=DEV).repeat_interleave(sigma)
    v = (u * sigma + torch.arange(sigma, device=DEV).repeat(n)) % n
    order = torch.randperm(n, device=DEV, generator=gen)
    return _csr(n, order[u], order[v], simple=False)


def _device_csr(case, seed):
    gen = _gen(seed)
    if case["graph"] == "rmat":
        return _rmat(case["scale"], case["factor"], gen)
    if case["graph"] == "er":
        return _er(case["n"], case["samples"], gen)
    if case["graph"] == "kmer":
        return _kmer(case["genome"], case["copies"], case["k"], gen)
    return _dbg(case["sigma"], case["k"], gen)


def _graph(off, nbr, name="graph"):
    def host(t):
        return t.to(torch.int32).cpu().numpy().view(np.uint32)
    return Graph(host(off), host(nbr), name)


def _tails(off):
    return torch.repeat_interleave(torch.arange(off.numel() - 1, device=DEV), off[1:] - off[:-1])


def _no_isolated(off, nbr, gen):
    """Every node without a neighbour gets one, chosen as often as it occurs in the lists."""
    n = off.numel() - 1
    lone = torch.nonzero(off[1:] == off[:-1]).reshape(-1)
    to = nbr[torch.randint(nbr.numel(), (lone.numel(),), device=DEV, generator=gen)]
    return _csr(n, torch.cat([_tails(off), lone]), torch.cat([nbr, to]))


def _mtx_text(off, nbr, edges, gen):
    """MatrixMarket pattern symmetric text of `edges` edges of a simple symmetric CSR, one
    "u v" line each."""
    n = off.numel() - 1
    u = _tails(off)
    once = torch.nonzero(u < nbr).reshape(-1)
    assert once.numel() >= edges
    once = once[torch.randperm(once.numel(), device=DEV, generator=gen)[:edges].sort()[0]]
    num = torch.stack([nbr[once] + 1, u[once] + 1])
    head = b"%%%%MatrixMarket matrix coordinate pattern symmetric\n%d %d %d\n" % (n, n, num.shape[1])
    width = 1 + sum((num >= 10**d).long() for d in range(1, 10))
    start = torch.cumsum(width.sum(0) + 2, 0)
    text = torch.full((int(start[-1]),), 32, dtype=torch.uint8, device=DEV)
    text[start - 1] = 10
    end = [start - width[1] - 3, start - 2]  # last digit of each number
    for i in range(2):
        x = num[i]
        for d in range(int(width[i].max())):
            has = width[i] > d
            text[(end[i] - d)[has]] = (48 + x % 10)[has].to(torch.uint8)
            x = torch.div(x, 10, rounding_mode="floor")
    return head + text.cpu().numpy().tobytes()


def _edges(case):
    """Lines of an ingest text: fewer than the distinct edges any seed gives."""
    return int(0.6 * (case["samples"] if case["graph"] == "er" else case["factor"] << case["scale"]))


# ---- the surrogate's network ------------------------------------------------------------
def _params(gen):
    """Weights as a trained network has them: W1[6][64], b1, W2[64][64], b2, W3[64], b3."""
    w = torch.randn(N_PARAMS, generator=gen, device=DEV, dtype=torch.float32)
    w[:384] *= 0.6
    w[384:448] *= 0.1
    w[448:4544] *= 0.15
    w[4544:4608] *= 0.1
    w[4608:4672] *= 0.2
    w[4672:] *= 0.1
    return w.cpu().numpy()


def _samples(count, gen):
    """Standardised inputs and target of a graph's nodes: correlated, heavy to the right."""
    z = torch.randn(count, 6, generator=gen, device=DEV)
    x = 0.7 * z[:, :1] + 0.5 * z + 0.1 * z**2
    y = x @ torch.tensor([0.1, 0.3, 0.2, 0.2, 0.1, 0.1], device=DEV) + 0.1 * torch.sin(3 * x[:, 0])
    return x.float().cpu().numpy(), y.float().cpu().numpy()


# ---- the contract -----------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "gradient":
        gen = _gen(seed)
        x, y = _samples(case["count"], gen)
        net = Surrogate(seed=1)
        net.set_params(params=_params(gen))
        return dict(kind=kind, net=net, x=x, y=y)
    if kind == "batch":
        rng = random.Random(case["sizes"])
        gen = _gen(seed)
        items = []
        for i in range(case["count"]):
            logn, deg, p = rng.uniform(case["lo"], case["hi"]), rng.uniform(4, 32), rng.randint(4, 8)
            if i < case["count"] // 2:
                n = int(round(2.0**logn))
                off, nbr = _er(n, int(n * deg / 2), gen)
            else:
                off, nbr = _rmat(int(round(logn)), max(1, int(round(deg / 2))), gen)
            items.append((_graph(off, nbr), p))
        return dict(kind=kind, batch=HyperBallBatch(items), count=case["count"])
    off, nbr = _device_csr(case, seed)
    if kind == "ingest":
        return dict(kind=kind, text=_mtx_text(off, nbr, _edges(case), _gen(seed + 1)))
    if kind == "walks":
        off, nbr = _no_isolated(off, nbr, _gen(seed + 2))
    g = _graph(off, nbr)
    del off, nbr
    torch.cuda.empty_cache()
    state = dict(case, g=g)
    if kind == "hyperball":
        state["h"] = HyperBall(g, case["p"], _run=False)
    elif kind == "walks":
        state["h"] = HyperBall(g, 4, _run=False)
        state["net"] = Surrogate(seed=1)
        state["net"].set_params(params=_params(_gen(seed + 1)))
    return state


def _results(h, out):
    got = {"iterations": h.get_iters()}
    if out == "accumulators":
        got["dist"], got["inv"] = h.geodesic_distances(), h.harmonic_geodesic_distances()
    if out in ("closeness", "all"):
        got["closeness"] = h.compute_closeness_centrality(True)
    if out in ("harmonic", "all"):
        got["harmonic"] = h.compute_harmonic_centrality(True)
    if out in ("lin", "all"):
        got["lin"] = h.compute_lins_centrality()
    return got


def run(state):
    kind = state["kind"]
    if kind == "new":
        with HyperBall(state["g"], state["p"]) as h:
            return _results(h, state["out"])
    if kind == "hyperball":
        state["h"].run(max_iters=state["iters"])
        return _results(state["h"], state["out"])
    if kind == "batch":
        state["batch"].run()
        return [state["batch"].accumulators(i) for i in range(state["count"])]
    if kind == "exact":
        cls = ExactClosenessCentrality if state["out"] == "closeness" else ExactHarmonicCentrality
        return cls(state["g"], True, sources=(0, state["sources"])).centralities()
    if kind == "ingest":
        g, info = read_mtx(state["text"])
        return {"offsets": g.offsets.view(np.int64), "neighbours": g.neighbours.view(np.int64),
                "entries": int(info.entries)}
    if kind == "walks":
        return state["net"].rank_walks(state["h"], state["passes"])[0]
    grad, loss = state["net"].gradient(state["x"], state["y"])
    return {"grad": grad, "loss": loss}


def exact(case, seed):
    """HyperBall's estimates are defined by f32 arithmetic and a table of empirical biases,
    so its centralities have no value in 64 bits; a CSR is whole numbers.  The exact
    centralities, the ranking and the gradient have one."""
    kind = case["kind"]
    if kind == "exact":
        off, nbr = _device_csr(case, seed)
        return _exact_centrality(off, nbr, case["sources"], case["out"])
    if kind == "gradient":
        gen = _gen(seed)
        x, y = _samples(case["count"], gen)
        w = _params(gen)
        return _exact_gradient(x, y, w)
    if kind == "walks":
        off, nbr = _no_isolated(*_device_csr(case, seed), _gen(seed + 2))
        return _exact_ranking(off, nbr, case["passes"], _params(_gen(seed + 1)))
    return None


def _exact_centrality(off, nbr, sources, out):
    """Level-synchronous searches, one column per source; the source itself is found again
    and counted, as the reference's searches do."""
    n = off.numel() - 1
    tail = _tails(off)
    result = torch.zeros(sources, dtype=torch.float64, device=DEV)
    step = max(1, min(1024, (1 << 31) // max(1, nbr.numel())))
    for s0 in range(0, sources, step):
        cols = min(step, sources - s0)
        seen = torch.zeros(n, cols, dtype=torch.bool, device=DEV)
        front = torch.zeros(n, cols, dtype=torch.float32, device=DEV)
        front[torch.arange(s0, s0 + cols, device=DEV), torch.arange(cols, device=DEV)] = 1
        total = torch.zeros(cols, dtype=torch.float64, device=DEV)
        level = 0
        while True:
            level += 1
            live = front.any(1)[tail]
            reached = torch.zeros_like(front).index_add_(0, nbr[live], front[tail[live]])
            new = (reached > 0) & ~seen
            count = new.sum(0).double()
            if not bool(count.any()):
                break
            seen |= new
            front = new.float()
            total += count * level if out == "closeness" else count / level
        reach = seen.sum(0).double()
        fine = (reach > 1) & (total > 0)
        result[s0:s0 + cols] = torch.where(fine, reach / torch.where(fine, total, 1.0), 0.0)
    return result


def _network(x, w):
    h = torch.nn.functional.gelu(x @ w[:384].view(6, 64) + w[384:448])
    h = torch.nn.functional.gelu(h @ w[448:4544].view(64, 64) + w[4544:4608])
    return h @ w[4608:4672] + w[4672]


def _exact_ranking(off, nbr, passes, w):
    """The network on the standardised logs of walk counts (sums of small integers: exact
    in 64 bits up to 2^53, rounded beyond)."""
    deg = (off[1:] - off[:-1]).double()
    tail = _tails(off)
    s = [deg]
    for _ in range(passes):
        s.append(torch.zeros_like(deg).index_add_(0, tail, s[-1][nbr]))
    top = torch.zeros_like(deg).index_reduce_(0, tail, deg[nbr], "amax")
    logs, lm = [torch.log1p(v) for v in s], torch.log1p(top)
    x = [*logs, lm, logs[-1] - logs[-2]] + ([logs[1] - logs[0]] if passes == 2 else [])
    x = torch.stack(x, 1)
    x = (x - x.mean(0)) / x.std(0, correction=0)
    w = torch.from_numpy(w).to(DEV).double()
    return torch.cat([_network(part, w) for part in x.split(1 << 18)])


def _exact_gradient(x, y, w):
    x, y = torch.from_numpy(x).to(DEV).double(), torch.from_numpy(y).to(DEV).double()
    w = torch.from_numpy(w).to(DEV).double().requires_grad_()
    loss = 0.0
    for a in range(0, y.numel(), 1 << 18):
        part = ((_network(x[a:a + (1 << 18)], w) - y[a:a + (1 << 18)]) ** 2).sum() / y.numel()
        part.backward()
        loss += float(part.detach())
    return {"grad": w.grad, "loss": loss}


def _size(case):
    """(nodes, arcs) one can expect of a case's graph."""
    if case["graph"] == "rmat":
        n = 1 << case["scale"]
        return n, 2 * case["factor"] * n * 0.95
    if case["graph"] == "er":
        return case["n"], 2 * case["samples"]
    if case["graph"] == "dbg":
        n = case["sigma"] ** case["k"]
        return n, 2 * n * case["sigma"]
    n = _kmer_nodes(case["genome"], case["copies"], case["k"])
    return n, 2 * n


def work(case):
    """Bytes one pass cannot do without: the inputs and the outputs once, and for
    HyperBall the CSR and the sketches (read and written) once in each iteration that
    still changes most of them -- about four where the graph's diameter is small, every
    one on chains."""
    kind = case["kind"]
    if kind == "gradient":
        # 2 flops per weight forward, 4 backward
        return {"bytes": case["count"] * 28 + N_PARAMS * 8, "flops": 6.0 * N_PARAMS * case["count"]}
    if kind == "batch":
        n = case["count"] * (2.0 ** case["hi"] - 2.0 ** case["lo"]) / ((case["hi"] - case["lo"]) * math.log(2))
        return {"bytes": 4 * n * (4 + 4 * 17 + 2 * 99 + 40) + 16 * n, "flops": 0}
    n, arcs = _size(case)
    if kind in ("new", "hyperball"):
        sweeps = case["iters"] if case["graph"] == "kmer" else min(4, case.get("iters") or 4)
        outputs = dict(all=3, accumulators=2).get(case["out"], 1)
        return {"bytes": sweeps * (4 * n + 4 * arcs + (2 << case["p"]) * n + 40 * n) + 8 * outputs * n, "flops": 0}
    if kind == "exact":
        return {"bytes": 4 * n + 4 * arcs + n * case["sources"] / 4 + 8 * case["sources"], "flops": 0}
    if kind == "ingest":
        digits = max(1, int(math.log10(n)) + 1)
        return {"bytes": _edges(case) * (2 * digits + 2 + 16) + 8 * n, "flops": 0}
    return {"bytes": case["passes"] * (4 * n + 4 * arcs + 16 * n) + 28 * n, "flops": 2.0 * N_PARAMS * n}
