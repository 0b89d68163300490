"""Timed work of the k-max-truss library, through its public entry points.

A user hands over an undirected graph -- pairs in host or device memory, an
edge-list file, a batch, or a stream of queries -- and gets (kmax, |T|), the
kmax-truss's edges or every edge's trussness back. The graphs are the
benchmark's families (Erdos-Renyi with a planted clique, R-MAT, Chung-Lu with
gamma 2.1, the batch and serving mixes) from the smallest serving query
(1,000 edges) to the largest single-GPU workload (500 M edges), sampled on the
device from the seed.
"""
from __future__ import annotations

import math
import tempfile
from pathlib import Path

import numpy as np
import torch

from kc_cuda_amd import Context, DeviceArray, Server, gen, solve_device_noalloc

DEV = "cuda"
RMAT = (0.57, 0.19, 0.19)   # the benchmark's quadrant probabilities (and the rest)
GAMMA = 2.1                 # the benchmark's power law
CHUNK = 1 << 26             # samples drawn at a time


# ------------------------------------------------------------------- cases --

def listed():
    return [
        # The smallest serving query: a call's fixed cost. From host memory,
        # with the edge set, as kmax_truss() and an interactive user ask for it.
        dict(name="tiny_host", kind="solve", graph="rmat", n=64, edges=1_000, clique=8, source="host", truss=True),
        # The benchmark's smallest workload (ER 16,384 vertices, average
        # degree 16, a planted 24-clique), pairs resident in device memory.
        dict(name="er16k_device", kind="solve", graph="er", n=16_384, edges=131_072, clique=24, source="device",
             truss=True),
        # The median serving query through the allocation-free entry point,
        # which tight loops call with pairs and results in device memory.
        dict(name="query_200k_noalloc", kind="noalloc", graph="chung_lu", n=40_000, edges=200_000, clique=33),
        # Per-edge trussness: the whole decomposition (kc_gpu -t) of a
        # power-law graph.
        dict(name="trussness_2m", kind="trussness", graph="chung_lu", n=200_000, edges=2_000_000, clique=30),
        # An edge list in no order, the way it falls out of a join or a crawl.
        dict(name="rmat18_shuffled", kind="solve", graph="rmat", n=1 << 18, edges=16 << 18, clique=0,
             source="shuffled", truss=True),
        # kc_gpu -f -o: an edge-list text file to (kmax, |T|) and the edge set.
        dict(name="tsv_rmat18", kind="tsv", graph="rmat", n=1 << 18, edges=16 << 18, clique=0),
        # An ordinary power-law graph on an odd number of vertices, with its edge set.
        dict(name="chung_lu_50m_edges", kind="solve", graph="chung_lu", n=4_999_999, edges=50_500_000, clique=60,
             source="device", truss=True),
        # The benchmark's R-MAT workload: scale 22, edge factor 16.
        dict(name="rmat22_device", kind="solve", graph="rmat", n=1 << 22, edges=16 << 22, clique=0, source="device",
             truss=False),
        # The benchmark's largest single-GPU workload: 50 M vertices, 505 M samples.
        dict(name="chung_lu_500m_edges", kind="solve", graph="chung_lu", n=50_000_000, edges=505_000_000, clique=60,
             source="device", truss=False),
        # An eighth of the benchmark's batch of independent graphs (64 to
        # 65,536 vertices, average degree 8 to 32, cliques of 4 to 40).
        dict(name="batch_512", kind="batch", count=512, n_min=64, n_max=65_536),
        # A burst of the benchmark's serving mix: lognormal sizes of median
        # 200,000 edges, R-MAT and Chung-Lu in turn, from host memory.
        dict(name="serve_48", kind="serve", count=48, median=200_000, sigma=1.5, cap=8_000_000),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "noalloc", "trussness", "tsv", "batch", "serve"])
    if kind == "batch":
        n_min = _log_uniform(rng, 64, 1024)
        return dict(kind=kind, count=_log_uniform(rng, 16, 512), n_min=n_min, n_max=_log_uniform(rng, n_min, 65_536))
    if kind == "serve":
        return dict(kind=kind, count=rng.randint(8, 64), median=_log_uniform(rng, 20_000, 200_000),
                    sigma=rng.uniform(0.5, 1.5), cap=8_000_000)
    top = dict(solve=64_000_000, noalloc=1_500_000, trussness=4_000_000, tsv=4_000_000)[kind]
    edges = _log_uniform(rng, 1_000, top)
    graph = rng.choice(["er", "rmat", "chung_lu"])
    # average degrees of the benchmark's graphs: 16 (ER), 32 (R-MAT), 10 to 20 (Chung-Lu)
    n = max(64, int(2 * edges / dict(er=rng.uniform(8, 32), rmat=32, chung_lu=rng.uniform(10, 20))[graph]))
    case = dict(kind=kind, graph=graph, n=n, edges=edges, clique=rng.randint(4, 64))
    if kind == "solve":
        small = edges < 10_000_000
        case |= dict(source=rng.choice(["host", "device", "shuffled"] if small else ["device", "shuffled"]),
                     truss=small or graph == "er" or rng.random() < 0.5)
    return case


# ------------------------------------------------------------------ graphs --

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(k, g):
    return torch.rand(k, generator=g, device=DEV, dtype=torch.float64)


def _endpoints_rmat(scale, k, g):
    """k endpoint pairs of R-MAT; scale: a number, or a tensor of one per pair."""
    top = int(scale if isinstance(scale, int) else scale.max())
    u = torch.zeros(k, dtype=torch.int64, device=DEV)
    v = torch.zeros_like(u)
    a, ab, abc = RMAT[0], RMAT[0] + RMAT[1], sum(RMAT)
    for lvl in range(top):
        x = torch.rand(k, generator=g, device=DEV)
        bu = x >= ab
        bv = ((x >= a) & ~bu) | (x >= abc)
        if not isinstance(scale, int):
            bu, bv = bu & (lvl < scale), bv & (lvl < scale)
        u |= bu.long() << lvl
        v |= bv.long() << lvl
    return u, v


def _endpoints_chung_lu(n, samples, k, g):
    """2k endpoints with probability proportional to i^(-1/(gamma-1)), capped
    at the square root of the sum (the continuous inverse of that law)."""
    a = 1.0 - 1.0 / (GAMMA - 1.0)
    # weights are w(x) = c x^(a-1) on [1, n] with integral 2 * samples
    c = 2.0 * samples * a / (n ** a - 1.0)
    cap = math.sqrt(2.0 * samples)
    x0 = min(float(n), max(1.0, (c / cap) ** (1.0 / (1.0 - a))))  # capped below x0
    head = cap * x0
    tail = c / a * (n ** a - x0 ** a)
    t = _rand(2 * k, g) * (head + tail)
    x = torch.where(t < head, t / cap, (x0 ** a + (t - head).clamp_min(0) * (a / c)).pow(1.0 / a))
    x = x.long().clamp_(0, n - 1)
    return x[:k], x[k:]


def _clique_keys(ids):
    i, j = torch.triu_indices(ids.numel(), ids.numel(), 1, device=DEV)
    a, b = ids[i], ids[j]
    return torch.minimum(a, b) << 32 | torch.maximum(a, b)


def _graph(graph, n, samples, clique, seed):
    """(m, 2) int32 pairs on the device, u < v, sorted, distinct, relabelled at random."""
    g = _gen(seed)
    perm = torch.randperm(n, generator=g, device=DEV)
    keys = []
    for at in range(0, samples, CHUNK):
        k = min(CHUNK, samples - at)
        if graph == "rmat":
            u, v = _endpoints_rmat(max(1, (n - 1).bit_length()), k, g)
        elif graph == "chung_lu":
            u, v = _endpoints_chung_lu(n, samples, k, g)
        else:
            u, v = (torch.randint(0, n, (k,), generator=g, device=DEV) for _ in range(2))
        ok = (u != v) & (u < n) & (v < n)
        u, v = perm[u[ok]], perm[v[ok]]
        keys.append(torch.minimum(u, v) << 32 | torch.maximum(u, v))
        del u, v, ok
    if clique:
        keys.append(_clique_keys(perm[torch.randperm(n, generator=g, device=DEV)[:clique]]))
    keys = torch.unique(torch.cat(keys))
    return torch.stack([(keys >> 32).int(), keys.int()], 1)


def _batch(case, seed):
    """Pairs of all graphs one after another, offsets and vertex counts: half
    ER, half R-MAT."""
    rng = np.random.default_rng(seed)
    count = case["count"]
    ns = np.exp(rng.uniform(np.log(case["n_min"]), np.log(case["n_max"]), count)).round().astype(np.int64)
    samples = (ns * rng.uniform(8, 32, count) / 2).astype(np.int64)
    rmat = torch.from_numpy(rng.random(count) < 0.5).to(DEV)
    cliques = torch.from_numpy(np.minimum(rng.integers(4, 41, count), ns)).to(DEV)
    g = _gen(seed)
    dn = torch.from_numpy(ns).to(DEV)
    start = torch.from_numpy(np.concatenate([[0], np.cumsum(ns)])).to(DEV)
    total = int(start[-1])
    vertex_of = torch.repeat_interleave(torch.arange(count, device=DEV), dn)
    # the vertices of each graph in a random order: perm[start + i]
    perm = torch.argsort(vertex_of.double() + _rand(total, g))
    of = torch.repeat_interleave(torch.arange(count, device=DEV), torch.from_numpy(samples).to(DEV))
    k = of.numel()
    scale = torch.ceil(torch.log2(dn.double())).long().clamp_min(1)
    ru, rv = _endpoints_rmat(scale[of], k, g)
    eu, ev = ((_rand(k, g) * dn[of]).long() for _ in range(2))
    r = rmat[of]
    u, v = torch.where(r, ru, eu), torch.where(r, rv, ev)
    ok = (u != v) & (u < dn[of]) & (v < dn[of])
    u, v = perm[start[of[ok]] + u[ok]], perm[start[of[ok]] + v[ok]]
    i, j = torch.triu_indices(40, 40, 1, device=DEV)
    q, at = torch.nonzero(j[None, :] < cliques[:, None], as_tuple=True)
    back = lambda x: perm[start[q + 1] - 1 - x]  # noqa: E731 - the last vertices of each order
    u, v = torch.cat([u, back(i[at])]), torch.cat([v, back(j[at])])
    keys = torch.unique(torch.minimum(u, v) << 32 | torch.maximum(u, v))
    u, v = keys >> 32, keys & 0xFFFFFFFF
    gid = vertex_of[u]
    offs = torch.zeros(count + 1, dtype=torch.int64, device=DEV)
    offs[1:] = torch.bincount(gid, minlength=count).cumsum(0)
    pairs = torch.stack([(u - start[gid]).int(), (v - start[gid]).int()], 1)
    return pairs, offs.cpu().numpy().astype(np.uint64), ns.astype(np.uint32)


def _host(pairs):
    return pairs.cpu().numpy().view(np.uint32)


def _serve_mix(case, seed):
    """The quantiles of the lognormal sizes, in an order of the seed's."""
    rng = np.random.default_rng(seed)
    normal = torch.distributions.Normal(0.0, 1.0)
    q = (torch.arange(case["count"], dtype=torch.float64) + 0.5) / case["count"]
    sizes = (case["median"] * torch.exp(case["sigma"] * normal.icdf(q))).clamp(1_000, case["cap"]).long().tolist()
    out = []
    for i, edges in enumerate(sizes):
        graph = ("rmat", "chung_lu")[i % 2]
        n = max(64, edges // 16 if graph == "rmat" else edges // 5)
        out.append((_host(_graph(graph, n, edges, int(rng.integers(8, 65)), int(rng.integers(1, 1 << 31)))), n))
    return [out[i] for i in rng.permutation(len(out))]


# --------------------------------------------------------------- the calls --

def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return dict(kind=kind, server=Server(slots=8), mix=_serve_mix(case, seed))
    if kind == "batch":
        pairs, offs, ns = _batch(case, seed)
        torch.cuda.synchronize()
        ctx = Context()
        run_ = ctx.batch(DeviceArray(ctx, pairs.data_ptr(), pairs.numel() * 4), offs, ns)
        return dict(kind=kind, ctx=ctx, run=run_, pairs=pairs)
    pairs = _graph(case["graph"], case["n"], case["edges"], case["clique"], seed)
    m, n = pairs.shape[0], case["n"]
    if kind == "tsv":
        folder = tempfile.TemporaryDirectory()
        path = Path(folder.name) / "graph.tsv"
        gen.write_tsv(path, _host(pairs))
        return dict(kind=kind, ctx=Context(), folder=folder, path=path, cap=_cap(case))
    if kind == "noalloc":
        state = dict(kind=kind, pairs=pairs, m=m, n=n, out=torch.empty((_cap(case), 2), dtype=torch.int32, device=DEV))
        torch.cuda.synchronize()
        return state
    ctx = Context()
    state = dict(kind=kind, ctx=ctx, m=m, n=n, truss=case.get("truss", False), cap=_cap(case))
    if case.get("source") == "host":
        return state | dict(host=_host(pairs))
    if case.get("source") == "shuffled":
        g = _gen(seed + 1)
        pairs = pairs[torch.randperm(m, generator=g, device=DEV)]
        flip = torch.rand(m, generator=g, device=DEV) < 0.5
        pairs = torch.where(flip[:, None], pairs.flip(1), pairs).contiguous()
    torch.cuda.synchronize()
    return state | dict(pairs=pairs, device=DeviceArray(ctx, pairs.data_ptr(), pairs.numel() * 4))


def _cap(case):
    """Rows of the edge buffers a caller keeps (a graph's edge count varies a
    little with the seed, a case's outputs have one shape)."""
    rows = case["edges"] + case["clique"] ** 2
    return rows if case["kind"] == "trussness" else min(rows, 1 << 20)


def _rows(edges, cap):
    """The sorted rows in an array of cap rows, the rest -1."""
    out = np.full((cap, edges.shape[1]), -1, dtype=np.int32)
    out[:len(edges)] = edges[:cap].view(np.int32)
    return out


def _answer(r):
    return dict(kmax=int(r.kmax), edges=int(r.truss_edges), max_core=int(r.max_core), k_hat=int(r.k_hat))


def run(state):
    kind = state["kind"]
    if kind == "serve":
        srv = state["server"]
        tickets = [srv.submit(pairs, n) for pairs, n in state["mix"]]
        done = [srv.wait(t) for t in tickets]
        return dict(kmax=np.array([r.kmax for r in done]), edges=np.array([r.truss_edges for r in done]),
                    status=np.array([r.status for r in done]))
    if kind == "batch":
        state["run"].solve()
        r = state["run"].result()
        return dict(kmax=r.kmax.view(np.int32), edges=r.edges.view(np.int64), status=r.status.view(np.int32))
    if kind == "tsv":
        r = state["ctx"].solve_tsv(state["path"])[0]
        return _answer(r) | dict(truss=_rows(state["ctx"].truss_edges(), state["cap"]))
    if kind == "noalloc":
        out = state["out"]
        r, size = solve_device_noalloc(0, state["pairs"].data_ptr(), state["m"], state["n"], out.data_ptr(), len(out))
        # its pairs come in no order: a set of edges, held as sorted keys
        keys = torch.full((len(out),), (1 << 62), dtype=torch.int64, device=DEV)
        t = out[:size].long()
        keys[:len(t)] = torch.sort(t[:, 0] << 32 | t[:, 1]).values
        return _answer(r) | dict(truss=keys)
    ctx = state["ctx"]
    if "host" in state:
        r = ctx.solve_pairs(state["host"], state["n"])
    else:
        r = ctx.solve_device(state["device"], state["m"], state["n"])
    if kind == "trussness":
        return _answer(r) | dict(trussness=_rows(ctx.trussness(), state["cap"]))
    return _answer(r) | (dict(truss=_rows(ctx.truss_edges(), state["cap"])) if state["truss"] else {})


def work(case):
    """The input read once (8 bytes a pair; 2 x 8 characters or so a line and
    two lines an edge for text) and the answers, which are small beside it.
    Integer work on sparse rows: no floating-point operations."""
    if case["kind"] == "batch":
        lo, hi = case["n_min"], case["n_max"]
        mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        return dict(bytes=8.0 * case["count"] * mean * 10, flops=0)
    if case["kind"] == "serve":
        mean = min(case["median"] * math.exp(case["sigma"] ** 2 / 2), case["cap"])
        return dict(bytes=8.0 * case["count"] * mean, flops=0)
    triples = 12.0 * case["edges"] if case["kind"] == "trussness" else 0.0
    return dict(bytes=(32.0 if case["kind"] == "tsv" else 8.0) * case["edges"] + triples, flops=0)


# ------------------------------------------------------------------- exact --

def _trussness(pairs):
    """Textbook peel: trussness of every edge {(u, v): t}."""
    nbr = {}
    for a, b in pairs:
        nbr.setdefault(a, set()).add(b)
        nbr.setdefault(b, set()).add(a)
    sup = {(a, b): len(nbr[a] & nbr[b]) for a, b in pairs}
    out, k = {}, 2
    while sup:
        stack = [e for e, s in sup.items() if s <= k - 2]
        while stack:
            a, b = stack.pop()
            if (a, b) in out:
                continue
            out[a, b] = k
            del sup[a, b]
            nbr[a].discard(b)
            nbr[b].discard(a)
            for w in nbr[a] & nbr[b]:
                for e in ((min(a, w), max(a, w)), (min(b, w), max(b, w))):
                    sup[e] -= 1
                    if sup[e] == k - 2:
                        stack.append(e)
        k += 1
    return out


def exact(case, seed):
    if case["kind"] in ("serve", "batch") or case["edges"] > 150_000:
        return None
    pairs = _host(_graph(case["graph"], case["n"], case["edges"], case["clique"], seed)).tolist()
    t = _trussness([tuple(p) for p in pairs])
    k = max(t.values(), default=0)
    top = sorted(e for e, x in t.items() if x == k) if k >= 3 else []
    out = dict(kmax=k if k >= 3 else 0, edges=len(top), max_core=None, k_hat=None)
    cap = _cap(case)
    if case["kind"] == "trussness":
        rows = [(a, b, x) for (a, b), x in sorted(t.items()) if x >= 3]
        return out | dict(trussness=_rows(np.array(rows, dtype=np.int32).reshape(-1, 3), cap))
    rows = np.array(top, dtype=np.int64).reshape(-1, 2)
    if case["kind"] == "noalloc":
        keys = np.full(cap, 1 << 62, dtype=np.int64)
        keys[:len(top)] = rows[:, 0] << 32 | rows[:, 1]
        return out | dict(truss=keys)
    return out | (dict(truss=_rows(rows.astype(np.int32), cap)) if case.get("truss", True) else {})
