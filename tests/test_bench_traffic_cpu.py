"""bench.py's choice of the step's kernel variant among those of a counter pass."""
from test_bench_cpu import _bench


def test_step_variant_is_chosen_by_its_arguments():
    b = _bench()
    name = "void srf::k_bp_tiled<{}>(srf::SegRec const*, srf::Item const*)"
    step, emap = name.format("true, false, false"), name.format("false, false, false")
    # whichever was dispatched first
    assert b._step_value({emap: 7.0, step: 5.0}, "k_bp_tiled") == 5.0
    assert b._step_value({step: 5.0, emap: 7.0, name.format("true, true, false"): 9.0}, "k_bp_tiled") == 5.0
    # none, another kernel's, or two names: no figure
    assert b._step_value({emap: 7.0}, "k_bp_tiled") is None
    assert b._step_value({step: 5.0}, "k_fp_tiled") is None
    assert b._step_value({step: 5.0, "other " + step: 6.0}, "k_bp_tiled") is None
