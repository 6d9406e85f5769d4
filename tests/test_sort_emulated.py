"""The sort on the CPU: the product's tl_sort.hip compiled for the host over the
HIP shim in tests/emu/ (emu_sort.cpp), one workgroup at a time with every lane
a thread, under AddressSanitizer, against std::sort and std::unique on seven
kinds of input.  emu_sort2 is built with small buckets and few of them a pass,
so that its inputs take two passes; emu_sort_full with more keys a bucket than
a workgroup holds, so that its inputs end in the radix sort."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emulators():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_sort", "_build/emu_sort2",
                    "_build/emu_sort_full"], check=True, capture_output=True)


@pytest.mark.parametrize("program,kind,sizes", [
    ("emu_sort", "u64", [2, 4096]),
    ("emu_sort", "i32", [4097]),
    ("emu_sort2", "i64", [3000]),
    ("emu_sort2", "u32", [4099]),
    ("emu_sort_full", "i64", [9000]),
])
def test_sort_emulated(emulators, program, kind, sizes):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), kind] + [str(n) for n in sizes],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(", right") == 7 * len(sizes), r.stderr[-4000:]
