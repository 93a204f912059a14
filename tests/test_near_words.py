"""The packed candidate words of the wide disc kernels on the CPU (tests/asan/near.cpp): right
for every number of candidates, and each word only ever accessed as a word -- the type sanitizer
reports stores or loads of its ids as 16-bit values, which -O3 may reorder against the word's."""

import importlib.util
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


def _build(typed):
    spec = importlib.util.spec_from_file_location("asan_build", HERE / "asan" / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod.build_near(typed)


@pytest.mark.parametrize("typed", [False, True])
def test_candidate_words(typed):
    exe = _build(typed)
    if exe is None:
        pytest.skip("the toolchain has no type sanitizer")
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, cwd="/tmp")
    assert r.returncode == 0 and "0 wrong" in r.stdout, r.stdout + r.stderr[-3000:]
    assert "type-aliasing-violation" not in r.stderr, r.stderr[:3000]
