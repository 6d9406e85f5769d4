"""Lookups that are given a perfect vEB layout with its own tables through the
other split's entry point, on the CPU as in test_tile_emulated.py: the search of
a perfect tree depends on its tables alone, whichever path answers it."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.mark.parametrize("program", ["emu_tile", "emu_part"])
@pytest.mark.parametrize("layout,kind,n", [("veb-as-mveb", "u64", 16383),
                                           ("mveb-as-veb", "i32", 16383),
                                           ("veb-as-mveb", "u32", 8191)])
def test_tables_decide(program, layout, kind, n):
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_tile", "_build/emu_part"], check=True,
                   capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), layout, kind, "1", "66001", str(n)],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(": 0 wrong") == 2, r.stderr[-4000:]
