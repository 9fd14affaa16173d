"""The library's host code over a fake device, under AddressSanitizer and
UndefinedBehaviorSanitizer (CPU only; tests/sanitize/host_check.cpp)."""
import os
import subprocess

import pytest

from test_sanitize import BUILD, SAN_ENV, built  # noqa: F401  (built: the fixture)


@pytest.mark.parametrize("name", ["failed_allocations", "server_during_run", "memory_beside_server", "enormous_set",
                                  "capped_runs", "all_waves_at_once", "batch_walks",
                                  "failed_host_allocations", "full_lists", "slices", "run_walks"])
def test_host(built, name):  # noqa: F811
    r = subprocess.run([os.path.join(BUILD, "host_check"), name], capture_output=True, text=True, timeout=120,
                       env=SAN_ENV)
    assert r.returncode == 0 and r.stdout.strip() == f"{name}: ok", r.stdout + r.stderr[-4000:]
