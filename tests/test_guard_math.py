"""Host-side check of the guarded divisions of compiled sweeps (no GPU)."""
from test_index_math import _build_run


def test_guarded_division_is_the_ieee_quotient_or_redone(tmp_path):
    assert "passed" in _build_run("guard_check", tmp_path)


def test_side_constants_in_range_of_const_div(tmp_path):
    assert "passed" in _build_run("constdiv_side_check", tmp_path)
