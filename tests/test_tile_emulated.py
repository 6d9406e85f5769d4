"""The lookups of large batches on the CPU: the product's tl_tile.hip compiled
for the host over the HIP shim in tests/emu/ (emu_tile.cpp), one workgroup at a
time with every lane a thread, on exactly sized buffers under AddressSanitizer.
Every answer is compared with the oracle's search, with distinct keys and with
keys that repeat.  emu_part is built with small ranges and few of them a pass,
so that the arrays here take two passes of the partition."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emulators():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_tile", "_build/emu_part"], check=True,
                   capture_output=True)


@pytest.mark.parametrize("program,layout,kind,b,sizes", [
    ("emu_tile", "bst", "u32", 1, [4096]),
    ("emu_tile", "btree", "i64", 16, [70003]),
    ("emu_tile", "btree", "u32", 7, [4097]),
    ("emu_tile", "mveb", "u64", 1, [70003]),
    ("emu_tile", "veb", "i32", 1, [70003]),
    ("emu_tile", "binary", "u64", 1, [70003]),
    ("emu_part", "bst", "u64", 1, [16384]),
    ("emu_part", "btree", "u64", 16, [30000]),
    ("emu_part", "btree", "i32", 1, [20001]),
    ("emu_part", "mveb", "i32", 1, [20003]),
    ("emu_part", "binary", "i64", 1, [16385]),
])
def test_lookups_emulated(emulators, program, layout, kind, b, sizes):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), layout, kind, str(b), "66001"]
                       + [str(n) for n in sizes], capture_output=True, text=True, timeout=900,
                       env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(": 0 wrong") == 2 * len(sizes), r.stderr[-4000:]
