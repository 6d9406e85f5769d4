"""Buckets of more keys than a workgroup of the sort's usual launch holds, on the
CPU as in test_sort_emulated.py: they are sorted by larger workgroups and the
radix sort is not needed.  emu_sort_large has buckets of 4096 to 8192 keys after
one pass, emu_sort2_large most of 512 to 1024, where 512 fit, after two."""
import os
import re
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.mark.parametrize("program,kind,n", [("emu_sort_large", "u64", 9000),
                                            ("emu_sort_large", "i32", 12289),
                                            ("emu_sort2_large", "u32", 40000)])
def test_large_buckets(program, kind, n):
    subprocess.run(["make", "-C", EMU, "-j4", "_build/" + program], check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), kind, str(n)], capture_output=True,
                       text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(" 0 fallback,") == 7, r.stderr[-4000:]
    assert len(re.findall(r" [1-9]\d* large, right", r.stderr)) >= 5, r.stderr[-4000:]
