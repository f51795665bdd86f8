"""The batch's packing ahead of its copies (host_ahead.h), built with g++ under ThreadSanitizer, and under
AddressSanitizer and UndefinedBehaviorSanitizer. CPU only; skipped where g++ lacks the sanitizers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("sanitize", ["thread", "address,undefined"])
def test_results_in_turn_and_few_at_once(tmp_path, sanitize):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "ahead_checks")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-pthread", f"-fsanitize={sanitize}",
                        os.path.join(ROOT, "tests", "host", "ahead_checks.cpp"), "-o", exe], capture_output=True, text=True)
    if r.returncode != 0 and ("sanitize" in r.stderr or "san" in r.stderr.split("cannot find")[-1][:20]):
        pytest.skip("g++ without sanitizer runtimes")
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer does not run on this kernel")
    assert r.returncode == 0 and "checked" in r.stdout, r.stdout + r.stderr
