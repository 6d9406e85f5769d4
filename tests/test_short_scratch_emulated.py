"""Permutations where the stash of the direct path or of the one-pass slides is
not to be had, on the CPU as in test_permute_emulated.py: the plan, which makes
do with less, does them."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.mark.parametrize("program,layout,width,n,scratch", [
    ("emu_permute", "bst", 4, 16385, 4096), ("emu_permute", "btree", 8, 10000, 4096),
    ("emu_permute", "mveb", 4, 20000, 4096), ("emu_permute", "veb", 8, 5000, 4096),
    ("emu_permute", "btree", 4, 300007, 1000000), ("emu_slide", "btree", 8, 3001, 1000)])
def test_short_scratch(program, layout, width, n, scratch):
    subprocess.run(["make", "-C", EMU, "-j4", "_build/" + program], check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", EMU_SCRATCH_MAX=str(scratch), EMU_B="7")
    r = subprocess.run([os.path.join(EMU, "_build", program), layout, str(width), str(n)],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count("0 wrong, inverse 0 wrong") == 1, r.stderr[-4000:]


def test_short_splitter_tables():
    """The sort where the splitters' tables are not to be had, but the radix sort's."""
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_sort2"], check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", EMU_SCRATCH_SLOT="5",
               EMU_SCRATCH_MAX="4000")
    r = subprocess.run([os.path.join(EMU, "_build", "emu_sort2"), "u64", "5000"],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(", right") == 7, r.stderr[-4000:]
