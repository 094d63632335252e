"""Placement workloads for timing the library: what a user of it has
it do, through its public entry points, from one read on a small tree to a
sequencing run on a 16S-scale one.

Every case is synthetic and made from its seed: a random Yule tree, sequences
evolved down it under the case's model (GTR or a 20-state matrix, four gamma
rates or Price-CAT's twenty), an alignment with 2% of gaps, and reads cut from
the leaves and inner nodes with 2% of substitutions, 0.3% of ambiguity codes
and 0.3% of inner gaps, as real reads have them.

Kinds of case (case["kind"]):
  place     Core.process_query for a batch: stage-1 ranking, baseball, Brent,
            keep, refinement, ratios (and with -p the posterior).  entry
            "records" is Placer.place with its Python records; "batch" is
            pp_place_batch, from host strings to host results; "resident" is
            pp_place_resident on uploaded queries and the results' download.
  optimize  Three_tax.optimize of (query, edge) jobs, Placer.optimize.
  rank      the reference tree's GLVs and the stage-1 scores of a batch.
  glv       a chain of the device GLV module's functions.
  twin      the per-call linear_c.c twins on host arrays.
"""
import ctypes as C
import math

import numpy as np

from pplacer_amd import glvm, linear, placer, refio
from pplacer_amd._lib import PP_EQUERY, PP_FP32, PP_FP64, Placement, Stats, check, lib

# discrete gamma, four categories, alpha = 0.5
GAMMA4 = (0.033388, 0.251916, 0.820268, 2.894428)
CAT20 = tuple(0.05 * (200.0 ** (k / 19.0)) for k in range(20))
LETTERS = {4: "ACGT", 20: "ARNDCQEGHILKMFPSTWYV"}
AMBIG = {4: "RYN", 20: "BZX"}
# states of the codes above that stand for more than one
AMBIG_STATES = {4: {"R": (0, 2), "Y": (1, 3), "N": (0, 1, 2, 3)},
                20: {"B": (2, 3), "Z": (5, 6), "X": tuple(range(20))}}

RECORD = np.dtype([("loc", "<i4"), ("pad", "<i4"), ("ml_ratio", "<f8"), ("log_like", "<f8"),
                   ("dist_bl", "<f8"), ("pend_bl", "<f8"), ("post_prob", "<f8"), ("marginal_prob", "<f8")])


def listed():
    return [
        # one read on a small tree: the smallest call, what an interactive
        # user or a service placing reads as they come waits for
        dict(name="one_read", kind="place", entry="records", states=4, model="gamma", precision="fp64",
             taxa=50, columns=1000, queries=1, lo=150, hi=300, pp=False),
        # one sample's reads on a small tree, the batched FP32 form
        dict(name="amplicons_fp32", kind="place", entry="batch", states=4, model="gamma", precision="fp32",
             taxa=50, columns=1000, queries=200, lo=150, hi=300, pp=False),
        # a lane of 16S reads on a 16S-scale reference, the plain FP64 form
        # from host strings to host results
        dict(name="reads_16s_fp64", kind="place", entry="batch", states=4, model="gamma", precision="fp64",
             taxa=2000, columns=1600, queries=10000, lo=100, hi=500, pp=False),
        # the same reference, a larger run, the FP32 form on resident reads
        dict(name="reads_16s_fp32", kind="place", entry="resident", states=4, model="gamma", precision="fp32",
             taxa=2000, columns=1600, queries=40000, lo=100, hi=500, pp=False),
        # full-length 16S sequences: longer than the register-resident classes
        dict(name="full_length_fp64", kind="place", entry="batch", states=4, model="gamma", precision="fp64",
             taxa=400, columns=1543, queries=257, lo=600, hi=1543, pp=False),
        # posterior probabilities (-p): nested integrals on top of a placement
        dict(name="posterior_fp64", kind="place", entry="batch", states=4, model="gamma", precision="fp64",
             taxa=300, columns=1200, queries=400, lo=100, hi=450, pp=True),
        # a Price-CAT reference package (FastTree's model), 20 categories
        dict(name="price_cat_fp64", kind="place", entry="batch", states=4, model="cat", precision="fp64",
             taxa=700, columns=1401, queries=2000, lo=100, hi=500, pp=False),
        # protein reads, both forms
        dict(name="protein_fp64", kind="place", entry="batch", states=20, model="gamma", precision="fp64",
             taxa=200, columns=397, queries=1500, lo=60, hi=397, pp=False),
        dict(name="protein_fp32", kind="place", entry="resident", states=20, model="gamma", precision="fp32",
             taxa=500, columns=400, queries=5000, lo=60, hi=400, pp=False),
        # a new reference tree and the ranking of its first reads
        dict(name="tree_and_ranking", kind="rank", states=4, model="gamma", precision="fp64",
             taxa=500, columns=1300, queries=1000, lo=100, hi=500),
        # a host that drives Glvm.Model itself: three evolves, products, a
        # pull, the likelihoods of one three-taxon tree
        dict(name="glv_chain", kind="glv", states=4, columns=1601),
        # a host that has only re-pointed its stubs: one likelihood and one
        # masked dot product per call from host arrays
        dict(name="twin_calls", kind="twin", states=20, columns=397),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("place",) * 8 + ("optimize", "optimize", "rank", "rank", "glv", "twin"))
    states = rng.choice((4, 4, 4, 20))
    if kind in ("glv", "twin"):
        return dict(kind=kind, states=states, columns=_log_int(rng, 40, 1601 if states == 4 else 500))
    model = rng.choice(("gamma", "gamma", "gamma", "cat"))
    precision = rng.choice(("fp64", "fp32"))
    columns = rng.randint(300, 1600) if states == 4 else rng.randint(80, 400)
    lo = rng.randint(40, columns // 3 + 20)
    hi = rng.randint(lo, columns)
    taxa = _log_int(rng, 12, 1200 if states == 4 else 250)
    case = dict(kind=kind, states=states, model=model, precision=precision, taxa=taxa, columns=columns, lo=lo, hi=hi)
    if kind == "rank":
        return dict(case, queries=_log_int(rng, 1, 2000))
    if kind == "optimize":
        return dict(case, queries=_log_int(rng, 1, 300))
    pp = states == 4 and precision == "fp64" and rng.random() < 0.2
    most = 300 if pp else 8000 if states == 4 else 1500
    return dict(case, entry=rng.choice(("records", "batch", "resident")), queries=_log_int(rng, 1, most), pp=pp)


# ---- inputs -------------------------------------------------------------------

def _tree(rng, taxa):
    """A random Yule tree with a trifurcating root in post-order numbering."""
    kids = {0: [1, 2, 3]}
    tips = [1, 2, 3]
    nxt = 4
    while len(tips) < taxa:
        k = int(rng.integers(len(tips)))
        kids[tips[k]] = [nxt, nxt + 1]
        tips[k] = nxt
        tips.append(nxt + 1)
        nxt += 2
    order, stack = [], [0]
    while stack:  # reversed pre-order with children pushed in order = post-order
        v = stack.pop()
        order.append(v)
        stack.extend(kids.get(v, ()))
    order.reverse()
    new = {v: i for i, v in enumerate(order)}
    children = [[new[c] for c in kids.get(v, ())] for v in order]
    names = [None if ch else "t%d" % i for i, ch in enumerate(children)]
    bl = rng.exponential(0.03 if taxa > 1000 else 0.06, len(children)) + 1e-6
    bl[-1] = 0.0
    return refio.Tree(children, bl, names)


def _model(rng, states):
    exch = rng.exponential(1.0, (states, states))
    exch = np.triu(exch, 1)
    exch = exch + exch.T
    statd = 0.9 * rng.dirichlet(np.ones(states)) + 0.1 / states
    return exch, statd / statd.sum()


def _expm(exch, statd, times):
    """P(t) for every t in times: expm of the normalised reversible rate matrix."""
    q = exch * statd[None, :]
    np.fill_diagonal(q, 0.0)
    np.fill_diagonal(q, -q.sum(1))
    q = q / -(statd * np.diag(q)).sum()
    d = np.sqrt(statd)
    a = d[:, None] * q / d[None, :]
    lam, u = np.linalg.eigh(0.5 * (a + a.T))
    e = np.exp(np.asarray(times)[..., None] * lam)
    return ((u / d[:, None]) * e[..., None, :]) @ (u * d[:, None]).T


class _Inputs:
    """Tree, model, alignment and reads of a case, as host arrays."""

    def __init__(self, case, seed):
        rng = np.random.default_rng([seed, case["taxa"], case["columns"], case["queries"], case["states"]])
        S, N = case["states"], case["columns"]
        self.tree = _tree(rng, case["taxa"])
        self.exch, self.statd = _model(rng, S)
        cat = case["model"] == "cat"
        self.rates = np.array(CAT20 if cat else GAMMA4)
        self.site_cat = rng.integers(0, len(self.rates), N) if cat else None
        site_cat = self.site_cat if cat else rng.integers(0, 4, N)
        G = self.tree.n_nodes
        # states of every node, parents (larger ids) first, a level at a time
        cum = np.cumsum(_expm(self.exch, self.statd, self.tree.bl[:, None] * self.rates[None, :]), axis=-1)
        st = np.empty((G, N), dtype=np.int8)
        st[G - 1] = np.minimum(np.searchsorted(np.cumsum(self.statd), rng.random(N)), S - 1)
        parent, depth = self.tree.parent(), self.tree.depth()
        for d in range(1, int(depth.max()) + 1):
            v = np.nonzero(depth == d)[0]
            c = cum[v[:, None], site_cat[None, :], st[parent[v]]]
            st[v] = np.minimum((rng.random((len(v), N, 1)) > c).sum(-1), S - 1)
        abet = np.frombuffer(LETTERS[S].encode(), np.uint8)
        self.leaf = {}
        for v in self.tree.leaves():
            row = abet[st[v]].copy()
            row[rng.random(N) < 0.02] = ord("-")
            self.leaf[v] = row.tobytes().decode()
        # reads
        Q = case["queries"]
        node = rng.integers(0, G - 1, Q)
        length = rng.integers(case["lo"], min(case["hi"], N) + 1, Q)
        start = (rng.random(Q) * (N - length + 1)).astype(np.int64)
        qid = np.repeat(np.arange(Q), length)
        col = np.arange(len(qid)) - np.repeat(np.cumsum(length) - length, length) + np.repeat(start, length)
        s = st[node[qid], col]
        u = rng.random(len(qid))
        s = np.where(u < 0.02, (s + rng.integers(1, S, len(qid))) % S, s)
        ch = abet[s]
        amb = np.frombuffer(AMBIG[S].encode(), np.uint8)
        pick = (u > 0.02) & (u < 0.023)
        ch = np.where(pick, amb[rng.integers(0, len(amb), len(qid))], ch)
        ch = np.where((u > 0.023) & (u < 0.026), ord("-"), ch).astype(np.uint8)
        rows = np.full((Q, N), ord("-"), np.uint8)
        rows[qid, col] = ch
        rows[np.arange(Q), start] = abet[st[node, start]]  # no read without an informative column
        self.rows = rows

    def strings(self):
        return [r.tobytes().decode() for r in self.rows]


def _placer(case, inp, tree=True):
    pl = placer.Placer(0)
    if case["model"] == "cat":
        pl.build_model_cat(inp.exch, inp.statd, inp.rates, inp.site_cat)
    else:
        pl.build_model(inp.exch, inp.statd, inp.rates)
    if tree:
        pl.set_tree(inp.tree, inp.leaf, case["columns"])
    return pl


def _glv_arrays(case, seed):
    """Three GLVs, a model and three branch lengths, and a site mask."""
    S, N = case["states"], case["columns"]
    rng = np.random.default_rng([seed, S, N])
    exch, statd = _model(rng, S)
    a = [rng.uniform(1e-3, 1.0, (4, N, S)) * np.exp2(-rng.integers(0, 30, N))[None, :, None] for _ in range(3)]
    e = [rng.integers(-40, 1, N).astype(np.int64) for _ in range(3)]
    bl = rng.uniform(0.01, 0.5, 3)
    mask = (rng.random(N) < 0.7).astype(np.uint16)
    mask[0] = 1
    return exch, statd, a, e, bl, mask


def prepare(case, seed):
    kind = case["kind"]
    precision = PP_FP32 if case.get("precision") == "fp32" else PP_FP64
    if kind == "glv":
        exch, statd, a, e, bl, mask = _glv_arrays(case, seed)
        pl = placer.Placer(0)
        pl.build_model(exch, statd, np.array(GAMMA4))
        x, y, z = (glvm.Glv.of_arrays(pl._ctx, u, v) for u, v in zip(a, e))
        return dict(kind=kind, pl=pl, m=glvm.GmixModel(pl), xyz=(x, y, z), bl=bl, mask=mask,
                    tmp=[x.mimic() for _ in range(4)])
    if kind == "twin":
        _, statd, a, _, _, mask = _glv_arrays(case, seed)
        return dict(kind=kind, statd=statd, xyz=a, mask=mask)
    inp = _Inputs(case, seed)
    if kind == "rank":
        return dict(kind=kind, pl=_placer(case, inp, tree=False), inp=inp, n=case["columns"],
                    queries=inp.strings(), precision=precision)
    pl = _placer(case, inp)
    if kind == "optimize":
        rng = np.random.default_rng([seed, 7])
        jobs = 4 * case["queries"]
        loc = rng.integers(0, inp.tree.n_nodes - 1, jobs)
        return dict(kind=kind, pl=pl, queries=inp.strings(), job_q=np.arange(jobs) // 4, loc=loc,
                    pend=np.full(jobs, 0.1), dist=inp.tree.bl[loc] / 2.0, precision=precision)
    Q = case["queries"]
    prefs = placer.default_prefs(calc_pp=True) if case["pp"] else placer.default_prefs()
    st = dict(kind=kind, entry=case["entry"], pl=pl, prefs=prefs, precision=precision, Q=Q, K=prefs.keep_at_most,
              pp=case["pp"])
    if case["entry"] == "records":
        st["queries"] = inp.strings()
        return st
    st.update(out=(Placement * (Q * prefs.keep_at_most))(), n_out=np.zeros(Q, np.int32),
              status=np.zeros(Q, np.int32))
    if case["entry"] == "resident":
        pl.upload_queries(inp.strings())
    else:
        st["text"] = inp.rows.tobytes()
    return st


# ---- one pass -----------------------------------------------------------------

def _ip(a):
    return a.ctypes.data_as(C.POINTER(C.c_int))


def _run_place(st):
    pl, Q, K = st["pl"], st["Q"], st["K"]
    names = ["ml_ratio", "log_like", "dist_bl", "pend_bl"] + (["post_prob", "marginal_prob"] if st["pp"] else [])
    if st["entry"] == "records":
        res, status, _ = pl.place(st["queries"], prefs=st["prefs"], precision=st["precision"])
        fields = (("like_weight_ratio", "likelihood", "distal_length", "pendant_length")
                  + (("post_prob", "marginal_like") if st["pp"] else ()))
        loc, val = np.zeros((Q, K), np.int32), np.zeros((len(fields), Q, K))
        for q, recs in enumerate(res):
            loc[q, :len(recs)] = [r.edge_num for r in recs]
            for i, f in enumerate(fields):
                val[i, q, :len(recs)] = [getattr(r, f) for r in recs]
        return dict(status=np.array(status), n_out=np.array([len(q) for q in res], np.int32), loc=loc,
                    **dict(zip(names, val)))
    out, n_out, status = st["out"], st["n_out"], st["status"]
    if st["entry"] == "batch":
        rc = lib().pp_place_batch(pl._ctx, Q, st["text"], C.byref(st["prefs"]), st["precision"], out,
                                  _ip(n_out), _ip(status), C.byref(Stats()))
        if rc != PP_EQUERY:  # some query failed: status says which
            check(rc, "place_batch")
    else:
        pl.place_resident(st["prefs"], st["precision"])
        check(lib().pp_results_download(pl._ctx, out, _ip(n_out), _ip(status)), "results_download")
    rec = np.frombuffer(out, RECORD).reshape(Q, K)
    kept = np.arange(K)[None, :] < n_out[:, None]
    return dict(status=status.copy(), n_out=n_out.copy(), loc=np.where(kept, rec["loc"], 0),
                **{f: np.where(kept, rec[f], 0.0) for f in names})


def run(st):
    kind = st["kind"]
    if kind == "place":
        return _run_place(st)
    if kind == "optimize":
        ll, pend, dist, calls, status = st["pl"].optimize(st["queries"], st["job_q"], st["loc"], st["pend"],
                                                          st["dist"], 1e-5, precision=st["precision"])
        ok = status == 0  # a failed job has no lengths
        return dict(status=status, calls=np.where(ok, calls, 0),
                    **{k: np.where(ok, v, 0.0) for k, v in (("ll", ll), ("pend", pend), ("dist", dist))})
    if kind == "rank":
        st["pl"].set_tree(st["inp"].tree, st["inp"].leaf, st["n"])
        return st["pl"].stage1_scores(st["queries"], precision=st["precision"])
    if kind == "glv":
        m, (x, y, z), (p, q, r, w) = st["m"], st["xyz"], st["tmp"]
        for dst, src, t in zip((p, q, r), (x, y, z), st["bl"]):
            m.evolve_into(dst, src, float(t))
        ll = m.log_like3(p, q, r)
        w.listwise_prod([p, q, r])
        w.perhaps_pull_exponent(-10)
        a, e = w.get()
        m.statd_pairwise_prod(r, p, q)
        like = np.array([ll, r.logdot(w), r.masked_logdot(w, st["mask"])])
        return dict(like=like, a=a, e=e)
    x, y, z = st["xyz"]
    util = np.empty(x.shape[1])
    ll = linear.ten_log_like3(st["statd"], x, y, z, util)
    like = np.array([ll, linear.ten_masked_logdot(x, y, st["mask"])])
    return dict(like=like, util=util, prod=linear.ten_pairwise_prod(None, x, y))


# ---- work and exact values ------------------------------------------------------

def work(case):
    """place / optimize: probes at about 230 pairs of lengths a query (10 edges
    of 23 probes, half of them distal) for baseball and as many again for the
    refinement, each the evolves it needs and one dot product; the bytes are
    the tree's rows of ten edges, the reads and the results.  rank: the scores
    written once, the GLVs and the log table once."""
    S = case["states"]
    R = 1 if case.get("model") == "cat" else 4
    N = case["columns"]
    if case["kind"] in ("glv", "twin"):
        v = 4 * N * S * 8
        if case["kind"] == "glv":
            return {"bytes": 5 * v, "flops": 3 * 2 * 4 * N * S * S + 12 * 4 * N * S}
        return {"bytes": 4 * v, "flops": 7 * 4 * N * S}
    Q = case["queries"]
    M = (case["lo"] + min(case["hi"], N)) / 2.0
    G = 2 * case["taxa"] - 2
    w = 4 if case["precision"] == "fp32" else 8
    if case["kind"] == "rank":
        return {"bytes": int(Q * (G - 1) * 8 + Q * N + 3 * G * N * R * S * 8 + 16 * G * N * w),
                "flops": int(Q * (G - 1) * M + 6 * 2 * G * N * R * S * S + 15 * 2 * G * N * R * S)}
    probe = 2 * R * S * S + 4 * R * S
    if case["kind"] == "optimize":
        return {"bytes": int(4 * Q * M * 2 * R * S * w + Q * N), "flops": int(4 * Q * 50 * M * probe)}
    probes = 460 + (7 * 460 if case["pp"] else 0)
    return {"bytes": int(Q * M * 10 * 2 * R * S * w + Q * N + Q * 7 * 48 + G * N * 16 * w),
            "flops": int(Q * M * (probes * probe + (G - 1)))}


def _lv_table(S):
    """Likelihood vectors by character, and whether it is informative."""
    lv = np.ones((256, S))
    inf = np.zeros(256, bool)
    for k, c in enumerate(LETTERS[S]):
        lv[ord(c)] = np.eye(S)[k]
        inf[ord(c)] = True
    for c, states in AMBIG_STATES[S].items():
        lv[ord(c)] = np.isin(np.arange(S), states)
        inf[ord(c)] = True
    return lv, inf


def _exact_rank(case, seed):
    """Felsenstein pruning with expm and per-site scaling: the likelihood of
    every read attached to every edge's middle by a branch of 0.1."""
    inp = _Inputs(case, seed)
    S, N = case["states"], case["columns"]
    tree, cat = inp.tree, case["model"] == "cat"
    G = tree.n_nodes
    if G * N * S * (1 if cat else 4) > 3e7 or case["queries"] * G * N > 3e9:
        return None
    lv, informative = _lv_table(S)
    rates = inp.rates[inp.site_cat][:, None] if cat else np.broadcast_to(inp.rates, (N, 4))  # [N, R]
    R = rates.shape[1]

    def evolve(x, t):  # x [N, R, S]
        p = _expm(inp.exch, inp.statd, t * inp.rates)
        if cat:
            return np.einsum("nij,nrj->nri", p[inp.site_cat], x)
        return np.einsum("rij,nrj->nri", p, x)

    def scaled(x, s):
        m = x.max(axis=(1, 2), keepdims=True)
        return x / m, s + np.log(m[:, 0, 0])

    down, up = [None] * G, [None] * G  # (partials [N, R, S], log scale [N])
    below = [None] * G                 # the node's partials at its parent's end
    for v in range(G):
        x, s = np.ones((N, R, S)), np.zeros(N)
        if not tree.children[v]:
            x = np.repeat(lv[np.frombuffer(inp.leaf[v].encode(), np.uint8)][:, None, :], R, axis=1)
        for c in tree.children[v]:
            x, s = x * below[c][0], s + below[c][1]
        down[v] = scaled(x, s)
        if v < G - 1:
            below[v] = (evolve(down[v][0], tree.bl[v]), down[v][1])
    up[G - 1] = (np.ones((N, R, S)), np.zeros(N))
    for v in range(G - 1, -1, -1):
        if not tree.children[v]:
            continue
        top = evolve(up[v][0], tree.bl[v]) if v < G - 1 else up[v][0]
        for c in tree.children[v]:
            x, s = top, up[v][1]
            for b in tree.children[v]:
                if b != c:
                    x, s = x * below[b][0], s + below[b][1]
            up[c] = scaled(x, s)
    chars = np.nonzero(informative)[0]
    rowof = np.zeros(256, np.int64)
    rowof[chars] = np.arange(len(chars))
    pend = np.repeat(lv[chars][:, None, :], R, axis=1)  # [C, R, S]
    p = _expm(inp.exch, inp.statd, 0.1 * inp.rates)
    if cat:
        pend = np.einsum("kij,crj->kcri", p, pend)[inp.site_cat]  # [N, C, 1, S]
    else:
        pend = np.broadcast_to(np.einsum("rij,crj->cri", p, pend), (N, len(chars), R, S))
    read, cols = np.nonzero(informative[inp.rows])  # every read has an informative column
    first = np.searchsorted(read, np.arange(case["queries"]))
    flat = cols * len(chars) + rowof[inp.rows[read, cols]]
    out = np.empty((case["queries"], G - 1))
    for v in range(G - 1):
        half = tree.bl[v] / 2.0
        x = inp.statd * evolve(down[v][0], half) * evolve(up[v][0], half)
        table = np.log(np.einsum("nrs,ncrs->nc", x, pend) / R) + (down[v][1] + up[v][1])[:, None]
        out[:, v] = np.add.reduceat(table.ravel()[flat], first)
    return out


def exact(case, seed):
    if case["kind"] == "rank":
        return _exact_rank(case, seed)
    if case["kind"] == "glv":
        exch, statd, a, e, bl, mask = _glv_arrays(case, seed)
        x, y, z = (np.einsum("rij,rnj->rni", _expm(exch, statd, t * np.array(GAMMA4)), u) for u, t in zip(a, bl))
        ln2 = math.log(2.0)
        ex = sum(e)
        ll = np.log((statd * x * y * z).sum((0, 2))).sum() - x.shape[1] * math.log(4.0) + ln2 * float(ex.sum())
        w = x * y * z
        k = np.frexp(w.max((0, 2)))[1]
        k = np.where(k < -10, k, 0)
        w = np.ldexp(w, -k[None, :, None])
        ew = (ex + k).astype(np.int64)
        er = e[0] + e[1]
        site = np.log((statd * x * y * w).sum((0, 2)) / 4.0) + ln2 * (er + ew)
        return dict(like=np.array([ll, site.sum(), site[mask > 0].sum()]), a=w, e=ew)
    if case["kind"] == "twin":
        _, statd, (x, y, z), _, _, mask = _glv_arrays(case, seed)
        util = (statd * x * y * z).sum((0, 2))
        dot = np.log((x * y).sum((0, 2)) / 4.0)[mask > 0].sum()
        return dict(like=np.array([np.log(util / 4.0).sum(), dot]), util=util, prod=x * y)
    # a placement or an optimisation is where a search stops within its
    # tolerance: the path's own answer, not a number that another method has
    return None
