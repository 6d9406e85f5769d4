"""Permutations of arrays that fit the stash whole (one copy, one pass of every
key to its slot) on the CPU, as in test_permute_emulated.py, at the edges of
its tiles and of every layout's shape; and the plans, which larger arrays take,
at the sizes of that file (TL_PERMUTE_PLAN keeps them for every size)."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emulator():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_permute"], check=True,
                   capture_output=True)
    return os.path.join(EMU, "_build", "emu_permute")


def run(emulator, layout, width, sizes, **env):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", **env)
    r = subprocess.run([emulator, layout, str(width)] + [str(n) for n in sizes],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count("0 wrong, inverse 0 wrong") == len(sizes), r.stderr[-4000:]


@pytest.mark.parametrize("layout", ["bst", "btree", "mveb", "veb"])
@pytest.mark.parametrize("width", [4, 8])
def test_direct_emulated(emulator, layout, width):
    run(emulator, layout, width,
        [2, 3, 15, 16, 17, 18, 255, 256, 257, 288, 289, 2047, 2048, 2049, 4912, 4913, 16385,
         65535, 65537])


@pytest.mark.parametrize("layout,width,sizes", [
    ("mveb", 8, [300007, 1048575]),
    ("mveb", 4, [300007]),
    ("bst", 8, [65536, 300007]),
    ("btree", 4, [300007]),
])
def test_plan_emulated(emulator, layout, width, sizes):
    run(emulator, layout, width, sizes, TL_PERMUTE_PLAN="1")
