"""What the tiles of the one-pass slides wait for, on the CPU (emu_slide_order.cpp):
every slot of the array that one tile stores to and another has to have loaded
before is among those the storing tile waits for, and the other has the earlier
ticket; perfect trees, trees with few leaves (whose level above moves straight
too) and with many, forward and inverse."""
import os
import random
import subprocess

import pytest

from test_slide_emulated import edges

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emulator():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_slide_order"], check=True,
                   capture_output=True)
    return os.path.join(EMU, "_build", "emu_slide_order")


@pytest.mark.parametrize("layout,b", [("bst", 1), ("btree", 1), ("btree", 2), ("btree", 3),
                                      ("btree", 7), ("btree", 16), ("btree", 63), ("btree", 300)])
def test_slide_order(emulator, layout, b):
    rng = random.Random(b)
    sizes = edges(b, 10000) + [rng.randint(b + 2, 12000) for _ in range(12)]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([emulator, layout, str(b)] + [str(n) for n in sizes], capture_output=True,
                       text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count(" 0 wrong") == 4 * len(sizes), r.stderr[-4000:]
