"""Memory safety of the series passes, the ones the kernels run on the
linspace grid (test_sanitized_host.py runs the walk passes of the CPU build):
tests/sanitized_series_run.py in a child process with the sanitizer runtime
preloaded."""

import os
import subprocess
import sys

import pytest

from .test_sanitized_host import ROOT, SAN, _runtime


@pytest.mark.skipif(not os.path.exists(SAN) or _runtime() is None, reason="sanitizer build or runtime missing")
def test_series_passes_under_address_and_ub_sanitizers():
    env = dict(os.environ, LD_PRELOAD=_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1", PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "sanitized_series_run.py")], env=env,
                       capture_output=True, text=True, timeout=900)
    report = (p.stdout + p.stderr)[-4000:]
    assert p.returncode == 0, report
    assert "runtime error" not in p.stderr and "AddressSanitizer" not in p.stderr, report
    assert "sanitized series runs clean" in p.stdout, report
