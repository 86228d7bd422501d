"""The rounding-tested Exp, Log and Tanh on the host (the sweep of
devmath_accuracy.cpp): they must give the reference forms' bit patterns, and
the f64 value each rounds must stay within its test's margin of the exact
function: 2^15, 2^12 and 2^13 f64 ulps, at least 2^-38, 2^-41 and 2^-40 of the
value.  The bound leaves the device's reciprocal (2^-46) and the library's f64
rounding their share."""
import pytest

from test_devmath_host import report  # noqa: F401  (the fixture)

MARGIN = {"exp_p": -38, "log_p": -41, "tanh_p": -40}


@pytest.mark.parametrize("name", sorted(MARGIN))
def test_rounding_tested_forms(report, name):  # noqa: F811
    row = report[name]
    assert row["samples"] > 1_000_000
    assert row["nan_mismatch"] == 0 and row["over_tol"] == 0 and row["ref_mismatch"] == 0, row
    assert row["max_rel_err_log2"] < MARGIN[name] - 1, row
    # flagged over all bit patterns: log's negative half, else rare
    assert row["flagged"] < (0.51 if name == "log_p" else 0.005), row


@pytest.mark.parametrize("name", ["exp_p", "tanh_p"])
def test_arguments_that_come_in_masses_are_decided(report, name):  # noqa: F811
    # masked scores whose exponential is subnormal, and NaN: a flag costs each
    # such element both forms, one element at a time
    assert report[name]["flagged_edge"] < 2.0 ** -10, report[name]


def test_log_of_a_flagged_argument(report):  # noqa: F811
    # the form that decides zeros, subnormals, negatives, infinities and NaN
    # by itself gives the reference form's bits everywhere
    row = report["log_rare"]
    assert row["nan_mismatch"] == 0 and row["over_tol"] == 0 and row["ref_mismatch"] == 0, row
