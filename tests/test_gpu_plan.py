"""The plan of a short pass (include/pplacer_hip.h, pp_launch_config) belongs to
the launch shape in force: it holds whenever a form's stream counts are the
defaults, however they came to be set, and ends where they are not.  The number
of baseball launches shows which plan a pass took.  A captured pass is replayed
only for the plan, model, tree and prior it was captured with."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SERIAL = {"pitch_streams": [0, 0], "refine_streams": [0, 0]}


def _print_case(name):
    print("\n[gpu case] %s" % name, flush=True)


@pytest.fixture(scope="module")
def reads():
    """A fresh context and reads of several masked-length classes."""
    from pplacer_amd import placer, synth
    wl = synth.make_workload("gtr50", seed=31, n_queries=48)
    pl, queries, _, _ = placer.setup_from_workload(wl)
    yield pl, queries
    pl.close()


@pytest.mark.parametrize("form", ["fp64", "fp32"])
def test_setting_the_reported_shape_changes_nothing(reads, form):
    from pplacer_amd import placer
    pl, queries = reads
    prec = placer.PP_FP64 if form == "fp64" else placer.PP_FP32
    prefs = placer.default_prefs(calc_pp=True)
    default = pl.launch_config()

    def launches(what):
        _print_case("short-pass plan, %s, %s" % (form, what))
        got, status, stats = pl.place(queries, prefs=prefs, precision=prec)
        return stats.n_pitch_launches, (got, list(status))

    try:
        merged, want = launches("fresh context")
        pl.set_launch_config(**default)
        assert launches("set to what get reports") == (merged, want)
        pl.set_launch_config(chunk=1000)
        assert launches("another chunk") == (merged, want)
        pl.set_launch_config(**dict(default, graph=1))
        for replay in range(3):
            _print_case("short-pass plan, %s, graph pass %d" % (form, replay))
            got, status, stats = pl.place(queries, prefs=prefs, precision=prec)
            assert (got, list(status)) == want and stats.n_pitch_launches == merged
        pl.set_launch_config(**dict(default, **SERIAL))
        n, got = launches("main stream")
        assert n > merged and got == want  # a launch per class
        pl.set_launch_config(**default)
        assert launches("defaults restored") == (merged, want)
    finally:
        pl.set_launch_config(**default)


def test_tuner_times_the_plan_in_force_first(reads, monkeypatch):
    from pplacer_amd import placer, tune
    pl, queries = reads
    default = pl.launch_config()
    prefs = placer.default_prefs()
    place, seen = pl.place_resident, []

    def recorded(*args):
        stats = place(*args)
        seen.append((pl.launch_config(), stats.n_pitch_launches))
        return stats

    _print_case("tuner on 48 reads")
    pl.upload_queries(queries)
    monkeypatch.setattr(pl, "place_resident", recorded)
    try:
        best, trials = tune.tune(pl, prefs, placer.PP_FP64, reps=1, pitch_streams=(2,), refine_streams=(),
                                 chunks=(), graphs=())
    finally:
        pl.set_launch_config(**default)
    # the untimed first pass and the first trial: the same shape, the same launches
    assert seen[0] == seen[1] and seen[0][0] == default == trials[0][0]
    assert seen[2][1] > seen[1][1]  # two streams asked for: a launch per class


def _graph_equals_eager(pl, queries, prefs, what):
    """A graph pass (captured or replayed), an eager one and a replay."""
    from pplacer_amd import placer
    got = []
    for graph in (1, 0, 1):
        _print_case("graph %d, %s" % (graph, what))
        pl.set_launch_config(graph=graph)
        rows, status, _ = pl.place(queries, prefs=prefs, precision=placer.PP_FP64)
        got.append((rows, list(status)))
    assert got[0] == got[1] and got[2] == got[1], what
    return got[1]


def test_graph_follows_the_prior(reads):
    """The prior's kind is an argument of a captured -p launch."""
    from pplacer_amd import placer
    pl, queries = reads
    prefs = placer.default_prefs(calc_pp=True)
    try:
        flat = _graph_equals_eager(pl, queries, prefs, "flat prior")
        pl.set_prior("uniform")
        uniform = _graph_equals_eager(pl, queries, prefs, "uniform prior")
        assert uniform != flat
        pl.set_prior("flat")
        assert _graph_equals_eager(pl, queries, prefs, "flat prior again") == flat
    finally:
        pl.set_prior("flat")
        pl.set_launch_config(graph=0)


def test_graph_follows_model_and_tree():
    """One context whose model and tree change between passes of the same
    queries: buffers keep their addresses, a captured pass must not be kept."""
    from pplacer_amd import placer, synth
    wl = synth.make_workload("gtr12", seed=5)
    small = synth.make_workload("gtr12", seed=6, n_taxa=9)
    pl, queries, statd, rates = placer.setup_from_workload(wl, premasked=False)
    prefs = placer.default_prefs()
    n = len(queries[0])
    try:
        four = _graph_equals_eager(pl, queries, prefs, "four rates")
        pl.build_model(wl.exch, statd, [1.0])
        pl.set_tree(wl.tree, wl.leaf_seqs(), n)
        one = _graph_equals_eager(pl, queries, prefs, "one rate")
        pl.build_model_cat(wl.exch, statd, [0.3, 1.0, 2.0], np.arange(n) % 3)
        pl.set_tree(wl.tree, wl.leaf_seqs(), n)
        cat = _graph_equals_eager(pl, queries, prefs, "three categories")
        pl.build_model(wl.exch, statd, rates)
        pl.set_tree(small.tree, small.leaf_seqs(), n)
        other = _graph_equals_eager(pl, queries, prefs, "another tree")
        pl.set_tree(wl.tree, wl.leaf_seqs(), n)
        assert _graph_equals_eager(pl, queries, prefs, "four rates again") == four
        assert len({str(r) for r in (four, one, cat, other)}) == 4
    finally:
        pl.close()


def test_graph_follows_the_longest_protein():
    """20 states: one class, whose capacity is the longest masked length."""
    from pplacer_amd import placer, synth
    wl = synth.make_workload("prot10", seed=4, n_queries=1, n_columns=300)
    pl, _, _, _ = placer.setup_from_workload(wl, premasked=False)
    prefs = placer.default_prefs()
    rows = list(wl.leaf_seqs().values())
    n = len(rows[0])
    try:
        pl.place(rows, prefs=prefs)  # the buffers' largest sizes from the start
        for m in (20, n, 20):
            got = _graph_equals_eager(pl, [r[:m] + "-" * (n - m) for r in rows], prefs, "proteins of %d sites" % m)
            assert all(s == 0 for s in got[1])
    finally:
        pl.close()


# around the classes' ends, the two-sites-a-lane classes, and (for four rates
# past 960 sites, else past 1,920) the streaming class
PLAN_LENGTHS = [30, 64, 65, 200, 300, 449, 700, 960, 961, 1200, 1500, 1569, 1900, 1920, 1921, 2100, 2200]


@pytest.mark.parametrize("form", ["fp64", "fp32"])
@pytest.mark.parametrize("model", ["four_rates", "one_rate", "cat20"])
def test_short_pass_plan_equals_main_stream(model, form):
    """All classes at once, the streaming one beside the others, in one chunk and
    in several: the results are the main stream's, bit for bit, with -p."""
    from pplacer_amd import placer
    from tests.test_gpu_streaming import long_workload, masked, rows_of
    wl = long_workload(22)
    wl.n_cats = 4 if model == "four_rates" else 1
    prec = placer.PP_FP64 if form == "fp64" else placer.PP_FP32
    prefs = placer.default_prefs(calc_pp=True, max_pitches=6, keep_at_most=3)
    pl, _, statd, _ = placer.setup_from_workload(wl)
    if model == "cat20":
        rng = np.random.default_rng(20)
        pl.build_model_cat(wl.exch, statd, np.sort(rng.uniform(0.05, 3.0, 20)), rng.integers(0, 20, 2200))
        pl.set_tree(wl.tree, wl.leaf_seqs(), 2200)
    try:
        rows = rows_of(wl)
        queries = [masked(rows[(i + 5 * k) % len(rows)], m) for k in range(3) for i, m in enumerate(PLAN_LENGTHS)]
        default = pl.launch_config()
        got = {}
        for name, shape in (("one chunk", default), ("four chunks", dict(default, chunk=13)),
                            ("main stream", dict(default, **SERIAL))):
            _print_case("gtr12 seed 22, 2,200 columns, %s, %s, %s" % (model, form, name))
            pl.set_launch_config(**shape)
            rows_, status, _ = pl.place(queries, prefs=prefs, precision=prec)
            got[name] = rows_, list(status)
    finally:
        pl.close()
    assert all(s == 0 for s in got["main stream"][1])
    assert got["one chunk"] == got["main stream"]
    assert got["four chunks"] == got["main stream"]
