"""The cohort walk's rounds in LDS, on the CPU: no wave draws into a place that
another wave may still have to read (tests/sanitize/rounds_check.cpp)."""
from test_sanitize import built, run  # noqa: F401  (built: the fixture)


def test_draws_wait_for_the_reads_of_other_waves(built):  # noqa: F811
    assert run("rounds_check").stdout.strip() == "rounds_check: ok"
