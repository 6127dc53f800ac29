"""Performance cases: update batches through the engine's public entry points.

A case is a labelled R-MAT graph (a=0.57, b=0.19, c=0.19), one or several
registered queries and an update batch.  One pass is what a window stream
does with a batch: its edges arrive and are matched (graph apply, Stage 1,
index maintenance, masks, matching, commit for every query), later they
expire (the same edges deleted: graph, Stage 1, index maintenance).  A pass
therefore ends where it began, and every pass does the same work.

Keys of a case:
  scale, degree, labels, zipf, initial
            the graph: 2^scale vertices, average degree, label count, Zipf
            exponent of the labels (0: uniform), share of the edges that is
            there before the stream
  batch     edges of the update batch
  queries   "shape:label,label,...;..." for a fixed query, or "walk:kind:size"
            (feed "host": a random-walk query sampled by the host pipeline)
  layout    main-index layout, "gamma" or "gpma"
  feed      "device": Stage 1 on the device over the resident graph;
            "host": the batch's keys come from the host CaLiG (Stage 2 alone,
            as the command line drivers feed it)
  step      "arrive": the batch arrives, is matched, expires;
            "slide": the batch arrives while as many older edges expire, then
            the other way round (two mixed batches);
            "destroyed": as "arrive", and the embeddings that the expiry
            destroys are counted too;
            "index": as "arrive" without matching, and the main index is read
            back after the commit
  serve     "plain": the queries one after another; "served": prepared
            concurrently and counted by one batched launch
"""
import numpy as np
import torch

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import HostSession, KeyBatch, Planner, synth_spec
from cgbdsm_amd.multi import QuerySet, QuerySpec

# Query shapes by kind and size (edges u < v in lexicographic order): trees,
# walks without chords ("sparse"), and shapes of average degree 3 or more.
SHAPES = {
    "tree4": "01 02 03",
    "tree5": "01 02 13 14",
    "tree6": "01 02 13 14 25",
    "tree9": "01 02 13 14 25 36 47 58",
    "sparse4": "01 12 23",
    "sparse5": "01 12 23 34",
    "sparse6": "01 03 12 23 34 45",
    "sparse9": "01 05 12 23 34 45 56 67 78",
    "dense4": "01 02 03 12 13 23",
    "dense5": "01 02 03 04 12 13 24 34",
    "dense6": "01 02 03 04 12 13 23 25 34 35",
}
A, B, C = 0.57, 0.19, 0.19


def listed():
    small = {"degree": 8.0, "labels": 4, "zipf": 0.0, "initial": 0.9, "layout": "gamma", "feed": "device",
             "step": "arrive", "serve": "plain"}
    s20 = {"scale": 20, "degree": 16.0, "labels": 16, "zipf": 1.2, "initial": 0.9, "layout": "gpma",
           "feed": "device", "step": "arrive", "serve": "plain"}
    # The 8-query mix: 5-dense, 5-tree, 5-sparse, 4-dense, 4-tree, 4-sparse, 6-dense, 6-tree.
    mix = ("dense5:0,1,2,3,4;tree5:1,0,2,3,1;sparse5:2,1,3,0,1;dense4:0,1,2,3;"
           "tree4:1,2,0,3;sparse4:0,2,1,3;dense6:1,2,3,4,5,6;tree6:3,1,2,0,4,1")
    return [
        # A few edges at a time on a small resident graph: latency only.
        dict(small, name="trickle-17-s11", scale=11, batch=17, queries="dense5:0,1,2,3,0"),
        # Stage 2 alone, fed by a host Stage 1 (the command line drivers), odd small batch.
        dict(small, name="host-keys-301-s14", scale=14, labels=8, batch=301, queries="walk:tree:5", feed="host"),
        # The whole 10 % stream of the scale-14 graph as one batch, fed by the host.
        dict(small, name="host-keys-6500-s14", scale=14, labels=8, batch=6500, queries="walk:sparse:6", feed="host",
             layout="gpma"),
        # A sliding window on a mid-size graph, insertions and deletions in every batch.
        dict(small, name="slide-5003-s17", scale=17, degree=12.0, labels=8, batch=5003, queries="sparse6:0,1,2,3,4,5",
             step="slide"),
        # Expiring edges whose destroyed embeddings are reported too.
        dict(small, name="destroyed-9001-s16", scale=16, labels=8, batch=9001, queries="dense4:0,1,2,3",
             step="destroyed", layout="gpma"),
        # Index maintenance without matching, the index read back (hand-over, checkpoint).
        dict(small, name="index-40009-s18", scale=18, degree=16.0, labels=8, batch=40009,
             queries="sparse9:0,1,2,3,4,5,6,7,0", step="index"),
        # A small batch on a large resident graph and a large index (interactive serving).
        dict(s20, name="serve-1999-s20", batch=1999, queries="tree5:0,1,2,1,3"),
        # The serving stream's median batch, default layout.
        dict(s20, name="serve-50000-s20", batch=50000, queries="sparse5:2,1,3,0,1", layout="gamma"),
        # The single-query stream: 100 000-edge batches, a 6-vertex dense query.
        dict(s20, name="dense6-100000-s20", batch=100000, queries="dense6:0,1,2,3,4,5"),
        # Several registered queries of uneven size over one batch, counted by one batched launch.
        dict(s20, name="mix8-served-100000-s20", batch=100000, queries=mix, serve="served"),
        # The index-maintenance graph: 80 % initial, batches of 1 M edges.
        dict(s20, name="stress-1000000-s22", scale=22, degree=32.0, labels=32, zipf=0.0, initial=0.8, batch=1000000,
             queries="tree5:0,1,2,3,4", layout="gamma"),
        # The multi-query headline graph with its kind of small frequent-label queries, plain.
        dict(s20, name="headline-250000-s21", scale=21, degree=24.0, batch=250000,
             queries="sparse5:2,0,0,1,0;sparse4:0,2,0,1;dense4:0,1,0,2;tree6:3,1,2,4,5,1"),
    ]


def label_shares(case):
    share = np.arange(1, case["labels"] + 1, dtype=np.float64) ** -case["zipf"]
    return share / share.sum()


def likely(case, shape, labels):
    """Whether the batch can be expected to make embeddings of the query: a tree or walk by their expected number on a
    graph without hubs (hubs only add to it), a dense shape by the graph and its labels."""
    share = label_shares(case)
    if shape.startswith("dense"):
        return case["batch"] >= 1000 and case["degree"] >= 12 and (case["labels"] <= 8 or case["zipf"] > 0) and \
            max(labels) < 5
    edges = len(SHAPES[shape].split())
    count = 2.0 ** case["scale"] * case["degree"] ** edges / 2.0 ** (case["scale"] * (edges - len(labels) + 1))
    for x in labels:
        count *= share[x]
    return edges * case["batch"] / (2.0 ** case["scale"] * case["degree"] / 2) * count >= 50


def draw(rng):
    scale = rng.randint(10, 20)
    case = {"scale": scale, "degree": float(rng.choice([6, 8, 12, 16, 24])),
            "labels": rng.choice([4, 8, 16] if scale <= 14 else [8, 16, 32]), "zipf": rng.choice([0.0, 1.2]),
            "initial": rng.choice([0.8, 0.9])}
    most = min(100000, int((1 << scale) * case["degree"] / 2 * (1 - case["initial"]) / 2))
    case["batch"] = max(3, int(16 * (most / 16.0) ** rng.random()))
    case["step"] = rng.choice(["arrive", "arrive", "arrive", "slide", "destroyed", "index"])
    case["layout"] = rng.choice(["gamma", "gpma"])
    host = scale <= 15 and case["step"] == "arrive" and rng.random() < 0.4
    case["feed"] = "host" if host else "device"
    many = rng.choice([1, 1, 2, 5, 8]) if case["step"] in ("arrive", "slide") and not host else 1
    case["serve"] = rng.choice(["plain", "served"]) if many > 1 else "plain"
    kinds = ["tree4", "tree5", "sparse4", "sparse5", "dense4", "dense5"]
    if scale <= 17:
        kinds += ["tree6", "sparse6", "dense6"]
    # Frequent labels of a Zipf graph make counts explode: large graphs take the others.
    first = 1 if case["zipf"] and scale > 16 else 0
    pool = list(range(first, min(case["labels"], first + 8)))

    def query():
        for _ in range(40):
            shape = rng.choice(["sparse9", "tree9"] if case["step"] == "index" and rng.random() < 0.5 else kinds)
            n = int(shape[-1])
            lab = rng.sample(pool, n) if n <= len(pool) and scale > 14 else [rng.choice(pool) for _ in range(n)]
            if case["step"] == "index" or likely(case, shape, lab):
                break
        else:
            shape, lab = rng.choice(["tree4", "sparse4"]), pool[:4]
            while not likely(case, shape, lab) and case["batch"] < most:
                case["batch"] = min(most, 2 * case["batch"] + 1)
        return shape + ":" + ",".join(str(x) for x in lab)

    if host:
        case["batch"] = max(case["batch"], min(most, 300))
        case["queries"] = "walk:%s:%d" % (rng.choice(["tree", "sparse"]), rng.randint(4, 6))
    else:
        case["queries"] = ";".join(query() for _ in range(many))
    return case


def parse(text):
    out = []
    for i, one in enumerate(text.split(";")):
        shape, lab = one.split(":")
        edges = [(int(e[0]), int(e[1])) for e in SHAPES[shape].split()]
        out.append(QuerySpec("%d-%s" % (i, shape), np.array([int(x) for x in lab.split(",")], dtype=np.int32),
                             np.array(edges, dtype=np.uint32)))
    return out


def graph_of(case, seed):
    """Labels (n), initial edges and `batch` stream edges (two batches for "slide") of the seeded graph."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=dev).manual_seed(seed * 7919 + 13)
    n = 1 << case["scale"]
    target = int(n * case["degree"] / 2)
    keys = torch.zeros(0, dtype=torch.int64, device=dev)
    while keys.numel() < target:
        m = int((target - keys.numel()) * 1.2) + 1024
        u = torch.zeros(m, dtype=torch.int64, device=dev)
        v = torch.zeros(m, dtype=torch.int64, device=dev)
        for _ in range(case["scale"]):
            p = torch.rand(m, generator=g, device=dev)
            u = 2 * u + (p >= A + B)
            v = 2 * v + (((p >= A) & (p < A + B)) | (p >= A + B + C))
        lo, hi = torch.minimum(u, v), torch.maximum(u, v)
        keys = torch.unique(torch.cat([keys, (lo * n + hi)[lo != hi]]))
    keys = keys[torch.randperm(keys.numel(), generator=g, device=dev)[:target]]
    weight = torch.arange(1, case["labels"] + 1, dtype=torch.float64, device=dev) ** -case["zipf"]
    cdf = torch.cumsum(weight / weight.sum(), 0)
    p = torch.rand(n, generator=g, device=dev, dtype=torch.float64)
    labels = torch.searchsorted(cdf, p).clamp(max=case["labels"] - 1)
    edges = torch.stack([keys // n, keys % n], 1).to(torch.int32).cpu().numpy()
    init = int(target * case["initial"])
    need = case["batch"] * (2 if case["step"] == "slide" else 1)
    return labels.to(torch.int32).cpu().numpy(), edges[:init], edges[init: init + need]


def prepare_host(case, seed):
    kind, size = case["queries"].split(":")[1:]
    spec = synth_spec(case["scale"], case["degree"], case["labels"], zipf_s=case["zipf"], seed=seed + 1,
                      initial_frac=case["initial"], query_size=int(size), query_kind=kind, query_seed=seed + 1)
    host = HostSession(spec=spec, threads=8)
    keys, dv, _, _ = host.initial_keys()
    eng = Engine(0)
    q = eng.query(host.query_tables)
    q.set_layout(case["layout"])
    card, avg = q.index_init(keys, dv)
    q.set_plan(host.make_plan(card, avg))
    new = host.next_batch(min(case["batch"], host.stream_edges_left()))
    none = np.zeros(0, dtype=np.uint64)
    old = KeyBatch(new.index, none, np.concatenate([new.ins, new.upd]), none, np.zeros_like(new.edge_ok), new.dv,
                   new.pairs, {})
    return {"case": case, "eng": eng, "q": q, "host": host, "new": new, "old": old}


def prepare(case, seed):
    if case["feed"] == "host":
        return prepare_host(case, seed)
    labels, initial, batch = graph_of(case, seed)
    eng = Engine(0)
    k = case["batch"]
    new, old = batch[:k], -batch[:k] - 1
    if case["step"] == "slide":
        initial = np.concatenate([initial, batch[k:]])
        stream = np.concatenate([new, -batch[k:] - 1, batch[k:], old])
    else:
        stream = np.concatenate([new, old])
    graph = eng.graph(labels, initial)
    graph.set_stream(stream)
    specs = parse(case["queries"])
    state = {"case": case, "eng": eng, "graph": graph, "ints": stream.size // 2}
    if len(specs) > 1:
        state["set"] = QuerySet(eng, graph, specs, layout=case["layout"], threads=8)
        return state
    sp = specs[0]
    planner = Planner(sp.labels, sp.edges)
    q = eng.query(planner.query_tables)
    q.set_layout(case["layout"])
    card, avg = q.calig_attach(graph, sp.labels)
    q.set_plan(planner.make_plan(card, avg))
    state["q"] = q
    if case["step"] == "index":
        # Where the program keeps the index that it reads back, with room for any graph of this kind.
        state["index"] = np.zeros(2 * int(index_entries(case, sp, labels.size)) + 65536, dtype=np.uint64)
    return state


def run(state):
    case, out = state["case"], []
    if case["feed"] == "host":
        q = state["q"]
        for keys in (state["new"], state["old"]):
            q.stage(keys)
            out += q.run_batch()[:2]
        return out
    for half in range(2):
        state["graph"].apply_range(half * state["ints"], state["ints"])
        if "set" in state:
            s = state["set"]
            out.append(s.run_served()[0] if case["serve"] == "served" else s.run_plain())
            continue
        q = state["q"]
        q.calig_update()
        if case["step"] == "destroyed":
            out += q.calig_match_deleted()
        if case["step"] != "index":
            out += q.run_batch()[:2]
            continue
        q.transfer_update_all()
        if q.transfer_update_index():
            q.batch_update_global_index()
        if half == 0:
            keys = q.export(0)
            state["index"][: keys.size] = keys
            state["index"][keys.size:] = 0
            out += [keys.size, state["index"]]
    return out


def index_entries(case, sp, n):
    """Main-index entries of a query if every label pair that matches is kept (an upper estimate)."""
    share = label_shares(case)
    pairs = float(sum(share[sp.labels[a]] * share[sp.labels[b]] for a, b in sp.edges))
    return 4 * pairs * n * case["degree"] / 2 * case["initial"]


def work(case):
    """The pass cannot do without: the batch's edges read (as stream ints, or as keys), the index entries of every
    query edge that they can match written on arrival and cleared on expiry, and the counts (or the index) written.
    Matching is a search: its list entries depend on the data and are not counted here."""
    share = label_shares(case)
    passes = 2 * (2 if case["step"] == "slide" else 1)
    total = 8.0 * case["batch"] * passes if case["feed"] == "device" else 0.0
    if case["feed"] == "host":
        size = int(case["queries"].split(":")[2])
        entries = (size - 1) * 2.0 * case["batch"] * float((share ** 2).sum())
        return {"bytes": 2 * (8 + 8) * entries + 8.0 * size, "flops": 0}
    n = 1 << case["scale"]
    for sp in parse(case["queries"]):
        pairs = float(sum(share[sp.labels[a]] * share[sp.labels[b]] for a, b in sp.edges))
        total += passes * 2.0 * case["batch"] * 2 * pairs * (8 + 4) + 8.0 * (sp.qe + 1)
        if case["step"] == "index":
            total += 8 * index_entries(case, sp, n)
    return {"bytes": total, "flops": 0}


def new_embeddings(labels, before, after, spec):
    """Embeddings of `spec` that edges of `after` without `before` make, by the largest query edge mapped to such an
    edge (int64 list; None when more than 2^24 partial embeddings are met).  before, after: sorted u * n + v keys of
    both directions."""
    n = labels.numel()
    fresh = after[~torch.isin(after, before)]
    counts = []
    for top, (a, b) in enumerate(spec.edges.tolist()):
        ok = (labels[fresh // n] == int(spec.labels[a])) & (labels[fresh % n] == int(spec.labels[b]))
        at = {a: 0, b: 1}
        rows = torch.stack([fresh[ok] // n, fresh[ok] % n], 1)
        while len(at) < spec.labels.size:
            x = next(x for x in range(spec.labels.size) if x not in at and
                     any((p in at and q == x) or (q in at and p == x) for p, q in spec.edges.tolist()))
            first = True
            for e, (p, q) in enumerate(spec.edges.tolist()):
                if x not in (p, q) or (q if p == x else p) not in at:
                    continue
                src = rows[:, at[q if p == x else p]]
                keys = after if e < top else before
                if first:
                    lo = torch.searchsorted(keys, src * n)
                    deg = torch.searchsorted(keys, src * n + n) - lo
                    if int(deg.sum()) > 1 << 24:
                        return None
                    at_row = torch.repeat_interleave(torch.arange(len(rows), device=rows.device), deg)
                    k = torch.arange(at_row.numel(), device=rows.device) - (torch.cumsum(deg, 0) - deg)[at_row]
                    v = keys[lo[at_row] + k] % n if at_row.numel() else at_row
                    ok = (labels[v] == int(spec.labels[x])) & (rows[at_row] != v[:, None]).all(1)
                    rows = torch.cat([rows[at_row], v[:, None]], 1)[ok]
                    first = False
                elif len(rows):
                    k = src * n + rows[:, -1]
                    rows = rows[keys[torch.searchsorted(keys, k).clamp(max=keys.numel() - 1)] == k]
            at[x] = len(at)
        # edges between the two first vertices and the others were checked as
        # each vertex came in; the anchor edge itself is new by choice
        counts.append(len(rows))
    return counts


def exact(case, seed):
    """Counts by joining edge tables, without the engine: small single-query device cases."""
    if case["feed"] == "host" or ";" in case["queries"] or case["scale"] > 17 or case["step"] == "index":
        return None
    labels, initial, batch = graph_of(case, seed)
    spec = parse(case["queries"])[0]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    lab = torch.from_numpy(labels).to(dev)
    n, k = lab.numel(), case["batch"]

    def keys(e):
        t = torch.from_numpy(e.astype(np.int64)).to(dev)
        return torch.cat([t[:, 0] * n + t[:, 1], t[:, 1] * n + t[:, 0]]).sort().values

    def made(kept, new):
        c = new_embeddings(lab, keys(kept), keys(np.concatenate([kept, new])), spec)
        return None if c is None else [sum(c), np.array(c, dtype=np.uint64)]

    zero = [0, np.zeros(len(spec.edges), dtype=np.uint64)]
    if case["step"] == "slide":
        parts = [made(initial, batch[:k]), made(initial, batch[k:])]
        return None if None in parts else parts[0] + parts[1]
    got = made(initial, batch)
    if got is None:
        return None
    return zero + got + got + zero if case["step"] == "destroyed" else got + zero
