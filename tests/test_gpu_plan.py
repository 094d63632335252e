"""The plan of a short pass (include/pplacer_hip.h, pp_launch_config) belongs to
the launch shape in force: it holds whenever a form's stream counts are the
defaults, however they came to be set, and ends where they are not.  The number
of baseball launches shows which plan a pass took."""
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
