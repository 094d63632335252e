"""Stage-2 kernels, the site-order sum and the log-sum twins at the sizes where
their work splits: masked lengths around whole waves, rounds and classes, the
sum's block sizes and the twins' 4,096-site pieces.

Likelihoods are compared with the oracle's at the branch lengths the job
reports, so that only the arithmetic is compared: FP64 within 1e-9 relative (the
bar of the parity tests); FP32 within 5e-6 a site (about 40 roundings of 2^-24
in a site's util, 2.4e-6, and as much again for its log)."""
import ctypes as C
import struct

import numpy as np
import pytest

from tests.helpers import oracle_setup, oracle_setup_cat

pytestmark = pytest.mark.gpu


def _print_case(name):
    print("\n[gpu case] %s" % name, flush=True)


def _masked(seq, m):
    """The first m informative columns of seq, the others gaps."""
    return seq[:m] + "-" * (len(seq) - m)


def _check_lengths(pl, core, tree, full, lengths, precision, tol):
    queries = [_masked(full, m) for m in lengths]
    n, loc = len(queries), (tree.n_nodes - 1) // 2
    ll, pend, dist, calls, st = pl.optimize(queries, list(range(n)), [loc] * n, [0.1] * n,
                                            [float(tree.bl[loc]) / 2] * n, 0.01, 2.0, precision)
    for j, m in enumerate(lengths):
        assert st[j] == 0, (m, st[j])
        want = core.log_like(queries[j], loc, pend[j], dist[j])
        assert abs(ll[j] - want) <= tol(m, want), (m, ll[j], want)


def _workload(name, seed):
    """The workload with one query, a leaf's gap-free row."""
    from pplacer_amd import synth
    wl = synth.make_workload(name, seed=seed, n_queries=1)
    wl.queries[:] = [("full", next(iter(wl.leaf_seqs().values())))]
    return wl


@pytest.mark.parametrize("form", ["fp64", "fp32"])
def test_nucleotide_masked_lengths(oracle, form):
    from pplacer_amd import placer
    lengths = [1, 63, 64, 65, 128, 129, 447, 448, 449, 960, 961, 1000]
    _print_case("gtr50 seed 12, masked lengths %s, %s" % (lengths, form))
    wl = _workload("gtr50", 12)
    model, pre, core, (full,) = oracle_setup(oracle, wl)
    pl = placer.setup_from_workload(wl)[0]
    try:
        tol = (lambda m, w: 1e-9 * abs(w)) if form == "fp64" else (lambda m, w: 5e-6 * m)
        _check_lengths(pl, core, wl.tree, full, lengths, placer.PP_FP64 if form == "fp64" else placer.PP_FP32, tol)
    finally:
        pl.close()


@pytest.mark.parametrize("n_cats", [1, 4, 5, 21, 32])
def test_price_cat_categories(oracle, n_cats):
    """A wave builds four categories' tables at a time: fewer, whole groups, a
    remainder, more groups than the workgroup has waves (two waves at 60 sites,
    the streaming form at 1,000)."""
    from pplacer_amd import placer
    _print_case("gtr50 seed 13, %d categories" % n_cats)
    wl = _workload("gtr50", 13)
    rng = np.random.default_rng(n_cats)
    rates = [float(r) for r in np.sort(rng.uniform(0.05, 3.0, n_cats))]
    o = oracle_setup_cat(oracle, wl, rates, rng.integers(0, n_cats, size=len(wl.ref_aln[0][1])))
    pl = placer.Placer(0)
    try:
        pl.build_model_cat(wl.exch, o["statd"], rates, o["site_cat"])
        pl.set_tree(wl.tree, o["leaf"], o["N"])
        _check_lengths(pl, o["core"], wl.tree, o["queries"][0], [60, 65, 300, 1000], placer.PP_FP64,
                       lambda m, w: 1e-9 * abs(w))
    finally:
        pl.close()


def test_protein_masked_lengths(oracle):
    """Rounds of 112 sites (448 worker lanes, four rates): G in registers, in LDS,
    in the scratch."""
    from pplacer_amd import placer
    lengths = [1, 16, 17, 111, 112, 113, 224, 225, 336, 337, 400]
    _print_case("prot500 seed 3, masked lengths %s" % lengths)
    wl = _workload("prot500", 3)
    model, pre, core, (full,) = oracle_setup(oracle, wl)
    pl = placer.setup_from_workload(wl)[0]
    try:
        _check_lengths(pl, core, wl.tree, full, lengths, placer.PP_FP64,
                       lambda m, w: 1e-9 * abs(w))
    finally:
        pl.close()


@pytest.mark.parametrize("n", [31, 32, 33, 36, 287, 288, 289, 543, 544, 545, 1055, 1056, 1057, 1088, 1152, 1216,
                               1567, 1568, 1569, 2017, 4064, 4095, 4096])
def test_site_order_sum_block_edges(n):
    """32 terms one by one, then 64 blocks of 4, 8, 16, 24 or n / 64."""
    from pplacer_amd import _lib
    _print_case("site-order sum, n=%d" % n)
    x = np.log(np.random.default_rng(n).uniform(1e-3, 1.0, n))
    want = 0.0
    for v in x:
        want += float(v)
    out = np.zeros(3)
    dp = C.POINTER(C.c_double)
    assert _lib.lib().pp_test_sequential_sum(x.ctypes.data_as(dp), n, out.ctypes.data_as(dp)) == 0
    assert struct.pack("<d", out[0]) == struct.pack("<d", want)


@pytest.mark.parametrize("S", [3, 4, 20])
@pytest.mark.parametrize("n", [1, 64, 65, 4096, 4097, 8300])
def test_log_sum_twin_lengths(oracle, S, n):
    """The stub's sum in site order, in pieces of 4,096 sites: bit for bit."""
    from pplacer_amd import linear
    _print_case("log-sum twin, %d states, %d sites" % (S, n))
    rng = np.random.default_rng(S * 10000 + n)
    x, y, z = (rng.random((n, S)) for _ in range(3))
    statd = rng.dirichlet(np.ones(S))
    mask = (rng.random(n) < 0.6).astype(np.uint16)
    mask[0] = 1
    assert linear.mat_log_like3(statd, x, y, z) == oracle.mat_log_like3(statd, x, y, z)
    assert linear.mat_masked_logdot(x, y, mask) == oracle.mat_masked_logdot(x, y, mask)
