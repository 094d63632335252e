"""Passes in short chunks spread the baseball and -p phases over streams until a
launch shape is set (include/pplacer_hip.h, pp_launch_config).  The results
must be those of the phases run one after another on the main stream, bit for
bit: 40 queries over several masked-length classes, with -p, placed by a fresh
context and again after the main-stream shape is set."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp64", "fp32"])
def test_forked_phases_equal_main_stream(form):
    from pplacer_amd import placer, synth
    print("\n[gpu case] forked phases, %s" % form, flush=True)
    prec = placer.PP_FP64 if form == "fp64" else placer.PP_FP32
    wl = synth.make_workload("gtr50", seed=31, n_queries=40)
    prefs = placer.default_prefs(calc_pp=True)
    pl, queries, _, _ = placer.setup_from_workload(wl)
    try:
        # gap-free queries beside the fragments: other masked-length classes
        queries = queries + ["".join(a if a != "-" else b for a, b in zip(q, queries[0][::-1]))
                             for q in queries[:8]]
        forked = pl.place(queries, prefs=prefs, precision=prec)
        pl.set_launch_config(pitch_streams=[0, 0], refine_streams=[0, 0])
        serial = pl.place(queries, prefs=prefs, precision=prec)
    finally:
        pl.close()
    assert list(forked[1]) == list(serial[1])
    assert forked[0] == serial[0]
