"""The sort's way out when buckets hold more keys than any workgroup takes, after
one pass and after two, on the CPU as in test_sort_emulated.py: the partitioned
keys, what the gaps hold and the splitters that were present give every distinct
key to the radix sort.  The two-pass program has 64 buckets of about 600 keys
where 512 fit, with the second pass's splitters among the keys; an input of one
value alone needs no way out."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.mark.parametrize("program,kind,n", [("emu_sort_full", "u32", 9000),
                                            ("emu_sort2_full", "u64", 40000),
                                            ("emu_sort2_full", "i32", 33001)])
def test_fallback_is_taken_and_right(program, kind, n):
    subprocess.run(["make", "-C", EMU, "-j4", "_build/" + program], check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", program), kind, str(n)], capture_output=True,
                       text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(", right") == 7, r.stderr[-4000:]
    assert r.stderr.count(" 1 fallback,") >= 5, r.stderr[-4000:]
