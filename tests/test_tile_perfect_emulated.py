"""Perfect trees and larger two-pass arrays in the large-batch lookups, on the CPU as
in test_tile_emulated.py."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.mark.parametrize("program,layout,kind,b,n", [
    ("emu_tile", "bst", "u32", 1, 65535), ("emu_tile", "btree", "i64", 16, 83520),
    ("emu_tile", "mveb", "u64", 1, 65535), ("emu_part", "mveb", "i32", 1, 70003),
    ("emu_part", "bst", "u32", 1, 65535), ("emu_part", "btree", "u64", 16, 83520),
    ("emu_part", "mveb", "u64", 1, 65535), ("emu_part", "veb", "i64", 1, 65535)])
def test_lookups_emulated(program, layout, kind, b, n):
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_tile", "_build/emu_part"], check=True,
                   capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), layout, kind, str(b), "66001", str(n)],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(": 0 wrong") == 2, r.stderr[-4000:]
