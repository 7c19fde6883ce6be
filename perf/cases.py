"""The calls that a user of this library times: graph searches of every size and row type, the
batched forms, and the entry-vertex network's training and inference.

listed() names the cases, draw() gives more of the same ranges; prepare() makes what a program holds
before the call (an uploaded index, a batch object or a network, and new queries), run() makes the
call, exact() restates its result in float64 torch and work() says what it cannot do without.

An index is uploaded once and serves many query batches, so prepare() keeps the two last indexes it
made (they depend on the case alone); the queries, budgets and minibatches come from the seed.
"""
import collections
import math

import numpy as np
import torch

import song_amd
from song_amd import learned

DEV = torch.device("cuda", 0)
DEGREE = 31  # neighbour slots of a graph row (32 words with the degree)
CENTERS = 1000


# ---------------------------------------------------------------- the cases

def listed():
    big = {"data": "mixture", "rows": 1_000_000, "dim": 128, "metric": "l2"}
    return [
        # one user's request answered on its own: host buffers in, ids and distances out
        {"name": "one query", "kind": "host", **big, "nq": 1, "pq": 100, "k": 10},
        # a serving loop's small fixed-size batch that may not allocate: latency of the longest query
        {"name": "serving batch", "kind": "noalloc", **big, "nq": 48, "pq": 128, "k": 10},
        # low-dimensional float vectors under cosine with the reference's arithmetic, its default budget
        {"name": "cosine 15k x 16", "kind": "device", "data": "uniform", "rows": 15_000, "dim": 16, "metric": "cos",
         "nq": 5000, "pq": 100, "k": 100},
        # the throughput benchmark: 10k queries at the budget that reaches recall@10 0.95
        {"name": "l2 10k queries", "kind": "device", **big, "nq": 10_000, "pq": 704, "k": 10},
        # an ordinary offline job at a moderate budget that keeps 100 results
        {"name": "l2 3001 queries", "kind": "device", **big, "nq": 3001, "pq": 200, "k": 100},
        # the search of the learned form: confident queries start near their result on BF16 rows, the
        # others run the full budget from vertex 0 on the float rows
        {"name": "learned batch", "kind": "learned", **big, "nq": 10_000, "pq": 704, "pq_learned": 128, "k": 10},
        # wide float descriptors with the default arithmetic (reference distances bit for bit)
        {"name": "wide rows exact", "kind": "device", "data": "factor", "rows": 120_000, "dim": 960, "metric": "l2",
         "nq": 1000, "pq": 200, "k": 100},
        # the same descriptors read as FP8 codes, the result list re-ranked with the float rows
        {"name": "wide rows fp8", "kind": "device", "data": "factor", "rows": 120_000, "dim": 960, "metric": "l2",
         "nq": 1000, "pq": 200, "k": 100, "storage": "fp8"},
        # requests with their own k and budget in one batch, inner product, replayed as a graph
        {"name": "uneven batch", "kind": "batch", "data": "unit", "rows": 500_000, "dim": 96, "metric": "ip",
         "nq": 40_000, "pq": 512, "k": 100},
        # the network's prediction for a query batch, and for a handful of queries
        {"name": "predict 10k", "kind": "infer", "batch": 10_000, "dim": 128, "hidden": 256, "classes": 4096},
        {"name": "predict 33", "kind": "infer", "batch": 33, "dim": 128, "hidden": 256, "classes": 4096},
        # a stretch of the network's training, then its parameters for a checkpoint
        {"name": "train 12 steps", "kind": "train", "batch": 1024, "dim": 128, "hidden": 256, "classes": 4096,
         "steps": 12},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "noalloc", "device", "device", "device", "batch", "learned", "infer", "train"])
    if kind == "infer":
        return {"kind": kind, "batch": _log(rng, 1, 10_000), "dim": _log(rng, 16, 256),
                "hidden": 16 * rng.randint(4, 24), "classes": _log(rng, 100, 4096)}
    if kind == "train":
        return {"kind": kind, "batch": _log(rng, 32, 1024), "dim": _log(rng, 16, 256),
                "hidden": 16 * rng.randint(4, 16), "classes": _log(rng, 100, 4096), "steps": rng.randint(2, 12)}
    data, metric = rng.choice([("mixture", "l2"), ("mixture", "l2"), ("uniform", "cos"), ("unit", "ip"),
                               ("factor", "l2")])
    if kind == "learned":
        data, metric = "mixture", "l2"
    dim = {"mixture": (32, 200), "uniform": (8, 100), "unit": (24, 160), "factor": (100, 960)}[data]
    rows = {"mixture": (20_000, 1_000_000), "uniform": (5000, 100_000), "unit": (20_000, 500_000),
            "factor": (5000, 120_000)}[data]
    c = {"kind": kind, "data": data, "rows": _log(rng, *rows), "dim": _log(rng, *dim), "metric": metric}
    if kind == "host":
        c.update(nq=_log(rng, 1, 64), pq=_log(rng, 16, 300))
    elif kind == "noalloc":
        c.update(nq=_log(rng, 1, 1000), pq=_log(rng, 16, 300))
    elif kind == "device":
        c.update(nq=_log(rng, 64, 1500 if data == "factor" else 10_000), pq=_log(rng, 16, 300 if data == "factor" else 704))
        if data in ("factor", "mixture") and rng.random() < 0.4:
            c["storage"] = rng.choice(["bf16", "fp8"])
    else:
        c.update(nq=_log(rng, 200, 1500 if data == "factor" else 10_000), pq=rng.choice([200, 300, 512, 704]))
    if kind == "learned":
        c["pq_learned"] = rng.choice([48, 64, 100, 128])
    c["k"] = min(rng.choice([1, 10, 10, 100]), c.get("pq_learned", c["pq"]), c["pq"])
    return c


# ---------------------------------------------------------------- vectors and graphs

def _gen(*key):
    s = 0
    for v in key:
        s = (s * 1_000_003 + int(v) + 17) % (1 << 62)
    return torch.Generator(device=DEV).manual_seed(s)


def _vectors(c, n, g, centers):
    """n vectors of the case's distribution (the same kinds as song_amd.datasets, made on the GPU)."""
    dim = c["dim"]
    if c["data"] == "mixture":
        lab = torch.randint(0, centers.shape[0], (n,), generator=g, device=DEV)
        x = centers[lab] + 20.0 * torch.randn((n, dim), generator=g, device=DEV)
        return x.round_().clamp_(0.0, 255.0) + 0.0
    if c["data"] == "uniform":
        return torch.rand((n, dim), generator=g, device=DEV) * 2.0 - 1.0
    x = torch.randn((n, 64 if c["data"] == "factor" else dim), generator=g, device=DEV)
    if c["data"] == "unit":
        return x / x.norm(dim=1, keepdim=True)
    x = x @ centers.T + 0.05 * torch.randn((n, dim), generator=g, device=DEV)
    return (x / 90.0 + 0.5).clamp_(0.0, 1.0)


def _centers(c):
    """What base and queries of a workload share: the mixture's centres, the factor model's loadings."""
    g = _gen(5, c["rows"], c["dim"])
    if c["data"] == "factor":
        return torch.randn((c["dim"], 64), generator=g, device=DEV)
    return torch.rand((CENTERS, c["dim"]), generator=g, device=DEV) * 255.0


def _nearest(a, b, metric, k):
    """Positions of the k nearest rows of b to each row of a."""
    out = []
    bn = (b * b).sum(1)
    for s in range(0, a.shape[0], 1 << 16):
        d = -(a[s:s + (1 << 16)] @ b.T) if metric != "l2" else bn - 2.0 * (a[s:s + (1 << 16)] @ b.T)
        out.append(torch.topk(d, k, dim=1, largest=False).indices)
    return torch.cat(out)


def _graph(x, metric):
    """Neighbour lists [n, 31] (-1 past the degree), the kind that an insertion build leaves: most of a
    vertex's links are near neighbours, a few lead to other regions.  Rows are grouped into cells
    around sampled rows (the hubs); a row links to its nearest rows in the cell, its hub and the next
    hubs; a hub links to near rows, near hubs and a few far ones."""
    n = x.shape[0]
    if metric != "l2":
        x = x / x.norm(dim=1, keepdim=True)
    g = _gen(7, n, x.shape[1])
    nh = max(8, n // 500)
    hubs = torch.randperm(n, generator=g, device=DEV)[:nh]
    near_hub = _nearest(x, x[hubs], metric, 5)
    out = torch.full((n, DEGREE), -1, dtype=torch.int64, device=DEV)
    out[:, 26:] = hubs[near_hub]
    cell = near_hub[:, 0].clone()
    cell[hubs] = torch.arange(nh, device=DEV)
    order = torch.argsort(cell, stable=True)
    ends = torch.cumsum(torch.bincount(cell, minlength=nh), 0).tolist()
    is_hub = torch.zeros(n, dtype=torch.bool, device=DEV)
    is_hub[hubs] = True
    start = 0
    for end in ends:
        m = order[start:end]
        start = end
        for s in range(0, m.numel(), 4096):
            r = m[s:s + 4096]
            d = (x[m] * x[m]).sum(1)[None, :] - 2.0 * (x[r] @ x[m].T)
            # no link to a hub or to itself here, and a total order among equal distances
            key = d.double() + torch.arange(m.numel(), device=DEV) * 1e-9
            key[:, is_hub[m]] = math.inf
            key[r[:, None] == m[None, :]] = math.inf
            v, i = torch.topk(key, min(26, m.numel()), dim=1, largest=False)
            out[r, :i.shape[1]] = torch.where(torch.isfinite(v), m[i], -1)
    hd = _nearest(x[hubs], x[hubs], metric, min(16, nh))
    far = torch.randint(0, nh, (nh, 3), generator=g, device=DEV)
    hd = torch.cat([hd, far], 1)
    own = torch.arange(nh, device=DEV)[:, None]
    dup = (hd == own) | ((hd[:, :, None] == hd[:, None, :]) & torch.ones(hd.shape[1], hd.shape[1], device=DEV).tril(-1).bool()).any(2)
    row = torch.cat([out[hubs, :DEGREE - hd.shape[1]], torch.where(dup, -1, hubs[hd])], 1)
    out[hubs] = row
    out = torch.where(out == torch.arange(n, device=DEV)[:, None], -1, out)
    return torch.gather(out, 1, torch.argsort((out < 0).to(torch.int8), dim=1, stable=True)), hubs


class _Held:
    """An uploaded index with the vectors and neighbour lists it was made from."""

    def __init__(self, c):
        self.centers = _centers(c)
        self.base = _vectors(c, c["rows"], _gen(3, c["rows"], c["dim"]), self.centers)
        self.nbrs, self.hubs = _graph(self.base, c["metric"])
        g = torch.zeros((c["rows"], DEGREE + 1), dtype=torch.int64, device=DEV)
        g[:, 0] = (self.nbrs >= 0).sum(1)
        g[:, 1:] = self.nbrs.clamp_min(0)
        self.index = song_amd.Index(self.base.cpu().numpy(), g.cpu().numpy().view(np.uint64), c["metric"])


_HELD = collections.OrderedDict()
_STREAM = []  # graph replays need a stream other than the default one; a program keeps one for its batches
_STORE = {"f32": song_amd.STORE_F32, "bf16": song_amd.STORE_BF16, "fp8": song_amd.STORE_FP8}


def _held(c):
    key = (c["data"], c["rows"], c["dim"], c["metric"])
    if key not in _HELD:
        while len(_HELD) >= 2:
            _HELD.popitem(last=False)
        _HELD[key] = _Held(c)
    _HELD.move_to_end(key)
    h = _HELD[key]
    if c["kind"] == "learned" or c.get("storage", "f32") != "f32":
        h.index.add_storage(_STORE[c.get("storage", "bf16")])
    return h


def _queries(c, seed, held):
    return _vectors(c, c["nq"], _gen(11, seed, c["nq"]), held.centers)


def _budgets(c, seed):
    """Per-query (pq, k) of the uneven batch: four budgets up to the largest, three result counts."""
    r = np.random.default_rng([seed, c["nq"]])
    pqs = [max(1, c["pq"] // 8), c["pq"] // 4, c["pq"] // 2, c["pq"]]
    pq = r.choice(np.asarray(pqs, dtype=np.int32), size=c["nq"])
    k = np.minimum(r.choice(np.asarray([1, 10, c["k"]], dtype=np.int32), size=c["nq"]), np.minimum(pq, c["k"]))
    return pqs, pq.astype(np.int32), k.astype(np.int32)


def _entries(c, seed, held, q):
    """Per-query (pq, start vertices) of the learned batch: about one query in 23 is not confident."""
    r = np.random.default_rng([seed, c["nq"], 1])
    low = torch.from_numpy(r.random(c["nq"]) < 0.044).to(DEV)
    near = held.hubs[_nearest(q, held.base[held.hubs], "l2", 4)].to(torch.int32)
    entry = torch.where(low[:, None], -1, near).to(torch.int32).contiguous()
    pq = torch.where(low, c["pq"], c["pq_learned"]).to(torch.int32)
    return low, entry, pq


# ---------------------------------------------------------------- prepare and run

def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind in ("infer", "train"):
        return _prepare_net(c, seed)
    h = _held(c)
    q = _queries(c, seed, h)
    s = {"case": c, "index": h.index, "q": q}
    if kind == "host":
        s["q"] = q.cpu().numpy()
        return s
    nq, k = c["nq"], c["k"]
    s["ids"] = torch.zeros((nq, k), dtype=torch.int32, device=DEV)
    s["dists"] = torch.zeros((nq, k), dtype=torch.float32, device=DEV)
    s["flags"] = torch.zeros(nq, dtype=torch.int32, device=DEV)
    if kind == "noalloc":
        s["mode"] = song_amd.resolve_mode(h.index, q)
    if kind == "batch":
        pqs, pq, kk = _budgets(c, seed)
        mode = song_amd.MODE_FP32
        s["batch"] = song_amd.Batch(h.index, [song_amd.tier(p) for p in pqs], nq, mode=mode)
        s["pq_arr"], s["k_arr"] = torch.from_numpy(pq).to(DEV), torch.from_numpy(kk).to(DEV)
        # entries past a query's own k are not written
        s["ids"].fill_(-1)
        s["dists"].fill_(math.inf)
    if kind == "learned":
        low, s["entry"], s["pq_arr"] = _entries(c, seed, h, q)
        tiers = [song_amd.tier(c["pq_learned"], storage=song_amd.STORE_BF16),
                 song_amd.tier(c["pq"], storage=song_amd.STORE_F32, waves_per_query=2)]
        s["batch"] = song_amd.Batch(h.index, tiers, nq, mode=song_amd.MODE_FP32)
        s["k_arr"] = torch.full((nq,), k, dtype=torch.int32, device=DEV)
    if "batch" in s:
        if not _STREAM:
            _STREAM.append(torch.cuda.Stream())
        s["stream"] = _STREAM[0]
    return s


def _net_inputs(c, seed):
    g = _gen(13, seed, c["batch"], c["dim"])
    width = (c["dim"] + 8 + 15) // 16 * 16
    steps = c.get("steps", 1)
    x = torch.randn((steps, c["batch"], width), generator=g, device=DEV)
    x[:, :, c["dim"] + 8:] = 0.0
    x = x.to(torch.bfloat16)
    labels = torch.randint(0, c["classes"], (steps, c["batch"]), generator=g, device=DEV).to(torch.int32)
    stop = 7.0 + torch.randn((steps, c["batch"]), generator=g, device=DEV)
    nbr = torch.randint(0, c["classes"], (c["classes"], 4), generator=g, device=DEV).to(torch.int32)
    nbr[:, 0] = torch.arange(c["classes"], device=DEV)
    return x, labels, stop, nbr


def _prepare_net(c, seed):
    x, labels, stop, nbr = _net_inputs(c, seed)
    net = learned.MLP(c["dim"] + 8, c["hidden"], c["classes"], max_batch=c["batch"] if c["kind"] == "train" else 1024,
                      seed=seed)
    xi = x.view(torch.int16)
    if c["kind"] == "infer":
        return {"case": c, "net": net, "x": xi[0].contiguous(), "nbr": nbr}
    return {"case": c, "net": net, "x": [v.contiguous() for v in xi], "labels": [v.contiguous() for v in labels],
            "stop": [v.contiguous() for v in stop]}


LR, STOP_WEIGHT = 1e-3, 0.05


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "host":
        return s["index"].search(s["q"], c["pq"], c["k"])
    if kind == "device":
        s["index"].search_device(s["q"], c["pq"], c["k"], s["ids"], s["dists"], s["flags"],
                                 storage=_STORE[c.get("storage", "f32")])
        return s["ids"], s["dists"], s["flags"]
    if kind == "noalloc":
        song_amd.search_device_noalloc(s["index"], s["q"], c["pq"], c["k"], s["ids"], s["dists"], s["flags"],
                                       mode=s["mode"])
        return s["ids"], s["dists"], s["flags"]
    if kind in ("batch", "learned"):
        with torch.cuda.stream(s["stream"]):
            s["batch"].run(s["q"], s["ids"], s["flags"], k=c["k"], pq_arr=s["pq_arr"], k_arr=s["k_arr"],
                           dists=s["dists"], entry=s.get("entry"), graph=True)
        return s["ids"], s["dists"], s["flags"]
    if kind == "infer":
        return s["net"].infer(s["x"], nbr=s["nbr"])
    for x, lab, st in zip(s["x"], s["labels"], s["stop"]):
        s["net"].train_step(x, lab, st, LR, STOP_WEIGHT)
    return s["net"].get_params()


# ---------------------------------------------------------------- float64 restatement

def _dist64(rows, q, metric):
    if metric == "l2":
        return ((rows - q) ** 2).sum(-1)
    dot = (rows * q).sum(-1)
    if metric == "ip":
        return -dot
    c2 = dot * dot / (rows * rows).sum(-1) / (q * q).sum(-1)
    return torch.where(dot < 0, c2, -c2)


def _search64(x, nbrs, metric, q, pq, entry=None):
    """The best-first search of every row of q in lockstep: the pq smallest expanded (distance, id) of
    each query.  Expands the smallest unexpanded candidate until the list is full and its largest
    distance is below the candidate's."""
    nq, n, inf = q.shape[0], x.shape[0], math.inf
    best_d = torch.full((nq, pq), inf, dtype=torch.float64, device=DEV)
    best_i = torch.full((nq, pq), -1, dtype=torch.int64, device=DEV)
    seen = torch.zeros((nq, n), dtype=torch.bool, device=DEV)
    live = torch.arange(nq, device=DEV)  # output row of each running query
    bd, bi = best_d.clone(), best_i.clone()
    if entry is None:
        entry = torch.zeros((nq, 1), dtype=torch.int64, device=DEV)
    else:
        entry = entry.long()
        entry = torch.where((entry < 0).all(1, keepdim=True) & (torch.arange(entry.shape[1], device=DEV) == 0), 0, entry)
    cap = 1024
    cd = torch.full((nq, cap + 1), inf, dtype=torch.float64, device=DEV)
    ci = torch.full((nq, cap + 1), -1, dtype=torch.int64, device=DEV)
    used = torch.zeros(nq, dtype=torch.int64, device=DEV)
    new, step, steps = entry, 0, torch.zeros(nq, dtype=torch.int64, device=DEV)
    while True:
        ok = new >= 0
        safe = new.clamp_min(0)
        fresh = ok & ~torch.gather(seen, 1, safe)
        seen.scatter_(1, safe, torch.gather(seen, 1, safe) | ok)
        d = torch.where(fresh, _dist64(x[safe].double(), q[:, None, :], metric), inf)
        at = used[:, None] + torch.cumsum(fresh, 1) - 1
        used = used + fresh.sum(1)
        if step % 16 == 0 and int(used.max()) + 32 * 17 > cap:
            grow = cap
            cd = torch.cat([cd[:, :cap], torch.full((cd.shape[0], grow + 1), inf, dtype=torch.float64, device=DEV)], 1)
            ci = torch.cat([ci[:, :cap], torch.full((ci.shape[0], grow + 1), -1, dtype=torch.int64, device=DEV)], 1)
            cap += grow
        at = torch.where(fresh, at, cap)
        cd.scatter_(1, at, d)
        ci.scatter_(1, at, safe)
        cd[:, cap] = inf
        now = cd.min(1).values
        pos = torch.where(cd == now[:, None], ci, n + 1).argmin(1, keepdim=True)
        top, tpos = bd.max(1)  # +inf while the list is not full
        done = (top < now) | torch.isinf(now)
        vid = torch.gather(ci, 1, pos)
        cd.scatter_(1, pos, inf)
        put = ~done & (now < top)
        bd.scatter_(1, tpos[:, None], torch.where(put, now, top)[:, None])
        bi.scatter_(1, tpos[:, None], torch.where(put[:, None], vid, torch.gather(bi, 1, tpos[:, None])))
        steps += ~done
        new = torch.where(done[:, None], -1, nbrs[vid[:, 0]])
        step += 1
        if step % 32 == 0:
            if bool(done.all()):
                break
            if float(done.float().mean()) > 0.2:
                best_d[live[done]], best_i[live[done]] = bd[done], bi[done]
                keep = ~done
                bd, bi, cd, ci, q, new, used, live = (t[keep] for t in (bd, bi, cd, ci, q, new, used, live))
                seen, steps = seen[keep], steps[keep]
    best_d[live], best_i[live] = bd, bi
    return best_d, best_i


def _best64(x, nbrs, c, q, pq, k, entry=None, coded=None):
    """Distances [nq, k] of the search in float64; coded: the rows as the search reads them, the list
    then ranked again with the rows themselves."""
    out = []
    step = max(1, min(5000, int(2e10 / x.shape[0])))
    for s in range(0, q.shape[0], step):
        qs = q[s:s + step].double()
        d, i = _search64(x if coded is None else coded, nbrs, c["metric"], qs, pq, None if entry is None else entry[s:s + step])
        if coded is not None:
            for b in range(0, qs.shape[0], 256):
                r = _dist64(x[i[b:b + 256].clamp_min(0)].double(), qs[b:b + 256, None, :], c["metric"])
                d[b:b + 256] = torch.where(i[b:b + 256] >= 0, r, math.inf)
        out.append(torch.sort(d, 1).values[:, :k])
    return torch.cat(out)


def _coded(x, storage):
    """The rows as the low-precision storage holds them."""
    amax = x.abs().amax(1, keepdim=True)
    if storage == "fp8":
        s = torch.where(amax > 0, amax / 448.0, 1.0)
        return (x / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).float() * s
    s = torch.where(amax > 0, torch.exp2(torch.frexp(amax).exponent.float()), 1.0)
    return (x / s).bfloat16().float() * s


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind in ("infer", "train"):
        return _exact_net(c, seed)
    h = _held(c)
    q = _queries(c, seed, h)
    if kind == "batch":
        _, pq, kk = _budgets(c, seed)
        d = torch.full((c["nq"], c["k"]), math.inf, dtype=torch.float64, device=DEV)
        for p in sorted(set(pq.tolist())):
            rows = torch.from_numpy(np.nonzero(pq == p)[0]).to(DEV)
            kr = min(p, c["k"])
            d[rows, :kr] = _best64(h.base, h.nbrs, c, q[rows], p, kr)
        col = torch.arange(c["k"], device=DEV)
        return None, torch.where(col < torch.from_numpy(kk).to(DEV)[:, None], d, math.inf), None
    if kind == "learned":
        low, entry, _ = _entries(c, seed, h, q)
        d = torch.empty((c["nq"], c["k"]), dtype=torch.float64, device=DEV)
        for rows, p in ((~low, c["pq_learned"]), (low, c["pq"])):
            if bool(rows.any()):
                d[rows] = _best64(h.base, h.nbrs, c, q[rows], p, c["k"], entry[rows])
        return None, d, None
    store = c.get("storage", "f32")
    d = _best64(h.base, h.nbrs, c, q, c["pq"], c["k"], coded=None if store == "f32" else _coded(h.base, store))
    return None, d, None


def _split(p, c, width):
    hid, no = c["hidden"], c["classes"] + 1
    out, o = [], 0
    for shape in ((hid, width), (hid,), (hid, hid), (hid,), (no, hid), (no,)):
        m = math.prod(shape)
        out.append(p[o:o + m].reshape(shape).clone())
        o += m
    return out


def _start_params(c, seed, width):
    """The network's initial parameters: He-uniform from a splitmix64 stream, biases zero."""
    hid, no, ind = c["hidden"], c["classes"] + 1, c["dim"] + 8
    parts = []
    at = 0
    for rows, cols, fan in ((hid, width, ind), (hid, hid, hid), (no, hid, hid)):
        i = np.arange(1 + at, 1 + at + rows * cols, dtype=np.uint64)
        at += rows * cols
        with np.errstate(over="ignore"):
            z = np.uint64(seed) + i * np.uint64(0x9E3779B97F4A7C15)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z ^= z >> np.uint64(31)
        u = (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
        w = ((2.0 * u - 1.0) * float(np.float32(math.sqrt(6.0 / fan)))).reshape(rows, cols)
        if cols == width and rows == hid and fan == ind:
            w[:, ind:] = 0.0
        parts += [w.reshape(-1), np.zeros(rows)]
    return torch.from_numpy(np.concatenate(parts)).to(DEV)


def _forward64(w, x):
    h1 = torch.relu(x @ w[0].T + w[1])
    h2 = torch.relu(h1 @ w[2].T + w[3])
    return h1, h2, h2 @ w[4].T + w[5]


def _exact_net(c, seed):
    x, labels, stop, nbr = _net_inputs(c, seed)
    width = x.shape[2]
    p = _start_params(c, seed, width)
    if c["kind"] == "infer":
        _, _, z = _forward64(_split(p, c, width), x[0].double())
        prob = torch.softmax(z[:, :-1], 1)
        conf = torch.gather(prob, 1, nbr[prob.argmax(1)].long()).sum(1).clamp_max(1.0)
        return None, conf, z[:, -1]
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for t in range(c["steps"]):
        w = _split(p, c, width)
        xb, lab, st = x[t].double(), labels[t].long(), stop[t].double()
        n = xb.shape[0]
        h1, h2, z = _forward64(w, xb)
        dz = torch.softmax(z[:, :-1], 1)
        dz[torch.arange(n, device=DEV), lab] -= 1.0
        dz = torch.cat([dz / n, (2.0 * STOP_WEIGHT * (z[:, -1] - st) / n)[:, None]], 1)
        dh2 = (dz @ w[4]) * (h2 > 0)
        dh1 = (dh2 @ w[2]) * (h1 > 0)
        g = torch.cat([(dh1.T @ xb).reshape(-1), dh1.sum(0), (dh2.T @ h1).reshape(-1), dh2.sum(0),
                       (dz.T @ h2).reshape(-1), dz.sum(0)])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - LR * (m / (1 - 0.9 ** (t + 1))) / ((v / (1 - 0.999 ** (t + 1))).sqrt() + 1e-8)
    return p


# ---------------------------------------------------------------- what a pass cannot do without

# distances of one search of budget pq on these graphs: (fixed, per entry of the budget), fitted to
# the means that the search's own counters give
_DISTANCES = {"mixture": (600.0, 1.5), "uniform": (450.0, 2.6), "unit": (700.0, 10.5), "factor": (600.0, 8.0)}


def _per_query(c, pq):
    """Expansions and distances of one search of budget pq."""
    fixed, each = _DISTANCES[c["data"]]
    return pq * 1.08 + 10.0, fixed + each * pq


def work(case):
    c = dict(case)
    if c["kind"] in ("infer", "train"):
        width = (c["dim"] + 8 + 15) // 16 * 16
        mul = c["hidden"] * (width + c["hidden"] + c["classes"] + 1)
        if c["kind"] == "infer":
            return {"bytes": 2 * mul + c["batch"] * (2 * width + 16), "flops": 2 * c["batch"] * mul}
        return {"bytes": c["steps"] * (mul * 24 + c["batch"] * (2 * width + 8)), "flops": 6 * c["steps"] * c["batch"] * mul}
    size = {"f32": 4 * c["dim"], "bf16": 2 * c["dim"] + 4, "fp8": c["dim"] + 4}

    def search(n, pq, store):
        e, d = _per_query(c, pq)
        return n * (d * size[store] + e * 4 * (DEGREE + 1) + 4 * c["dim"]), n * d * 3 * c["dim"]

    if c["kind"] == "batch":
        parts = [search(c["nq"] / 4, p, "f32") for p in (max(1, c["pq"] // 8), c["pq"] // 4, c["pq"] // 2, c["pq"])]
    elif c["kind"] == "learned":
        parts = [search(0.956 * c["nq"], c["pq_learned"], "bf16"), search(0.044 * c["nq"], c["pq"], "f32")]
    else:
        parts = [search(c["nq"], c["pq"], c.get("storage", "f32"))]
    return {"bytes": sum(p[0] for p in parts) + c["nq"] * c["k"] * 8, "flops": sum(p[1] for p in parts)}
