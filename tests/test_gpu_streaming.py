"""The streaming form of stage 2 (masked lengths past the register-resident
classes) and the classes of two sites a lane, for every 4-state model: four
rates, one rate and Price-CAT.  With one GLV row a site the streaming form
begins at 1,921 sites, so the alignment has 2,200 columns; the site-order sum
takes blocks of n / 64 terms from 1,569 sites on, and the streaming kernels run
more waves (16) than 20 categories have table groups.

Likelihoods are compared with the oracle's at the branch lengths the job
reports: FP64 within 1e-9 relative (the bar of the parity tests); FP32 within
5e-6 a site (about 40 roundings of 2^-24 in a site's util, 2.4e-6, and as much
again for its log)."""
import numpy as np
import pytest

from tests.helpers import oracle_setup, oracle_setup_cat

pytestmark = pytest.mark.gpu

LENGTHS = [64, 960, 961, 1408, 1409, 1568, 1569, 1919, 1920, 1921, 2100, 2200]


def rows_of(wl):
    """The leaves' rows, which hold no gaps."""
    return list(wl.leaf_seqs().values())


def long_workload(seed):
    """12 taxa, 2,200 columns, one full-length query."""
    from pplacer_amd import synth
    wl = synth.make_workload("gtr12", seed=seed, n_queries=1, n_columns=2200)
    wl.queries[:] = [("full", rows_of(wl)[0])]
    return wl


def masked(seq, m):
    """The first m informative columns of seq, the others gaps."""
    return seq[:m] + "-" * (len(seq) - m)


@pytest.mark.parametrize("form", ["fp64", "fp32"])
@pytest.mark.parametrize("model", ["four_rates", "one_rate", "cat1", "cat20", "cat32"])
def test_long_rows_match_oracle(oracle, model, form):
    from pplacer_amd import placer
    print("\n[gpu case] gtr12 seed 21, 2,200 columns, %s, %s, lengths %s" % (model, form, LENGTHS), flush=True)
    wl = long_workload(21)
    if model.startswith("cat"):
        n_cats = int(model[3:])
        rng = np.random.default_rng(n_cats)
        rates = [float(r) for r in np.sort(rng.uniform(0.05, 3.0, n_cats))]
        o = oracle_setup_cat(oracle, wl, rates, rng.integers(0, n_cats, size=2200))
        core, full = o["core"], o["queries"][0]
        pl = placer.Placer(0)
        pl.build_model_cat(wl.exch, o["statd"], rates, o["site_cat"])
        pl.set_tree(wl.tree, o["leaf"], o["N"])
    else:
        wl.n_cats = 4 if model == "four_rates" else 1
        _, _, core, (full,) = oracle_setup(oracle, wl)
        pl = placer.setup_from_workload(wl)[0]
    try:
        assert len(full) == 2200
        queries = [masked(full, m) for m in LENGTHS]
        n, loc = len(queries), (wl.tree.n_nodes - 1) // 2
        ll, pend, dist, calls, st = pl.optimize(queries, list(range(n)), [loc] * n, [0.1] * n,
                                                [float(wl.tree.bl[loc]) / 2] * n, 0.01, 2.0,
                                                placer.PP_FP64 if form == "fp64" else placer.PP_FP32)
        for j, m in enumerate(LENGTHS):
            assert st[j] == 0, (m, st[j])
            want = core.log_like(queries[j], loc, pend[j], dist[j])
            tol = 1e-9 * abs(want) if form == "fp64" else 5e-6 * m
            assert abs(ll[j] - want) <= tol, (m, ll[j], want)
    finally:
        pl.close()
