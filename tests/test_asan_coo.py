"""The COO radius graph (coo.hip) on the CPU under AddressSanitizer and UBSan
(tests/asan/coo.cpp): exact buffers, odd sizes, edges equal to a plain loop's, and an error of
the wait that is not left for the next call to find."""

import importlib.util
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_edges_clean_under_sanitizers():
    spec = importlib.util.spec_from_file_location("asan_build", HERE / "asan" / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    r = subprocess.run([str(mod.build_coo())], capture_output=True, text=True, timeout=600, cwd="/tmp")
    assert r.returncode == 0 and "0 case(s) failed" in r.stdout, r.stdout + r.stderr[-3000:]
    assert "ERROR: AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr
