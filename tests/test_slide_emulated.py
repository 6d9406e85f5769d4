"""One-pass permutations of BSTs and B-trees (leaves straight to their slots,
internal keys through the stash) on the CPU, as in test_permute_emulated.py, in
tiles of 512 keys: perfect trees, trees with few leaves (whose level above goes
straight too) and with many, partial leaves."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emulator():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_slide"], check=True,
                   capture_output=True)
    return os.path.join(EMU, "_build", "emu_slide")


def edges(b, top):
    k, sizes = b + 1, {b + 1, b + 2, 511, 512, 513, 1024, 1025, 3001}
    p = k
    while p <= top:
        for d in (-1, 0, 1, b - 1, b, k, p // k - 1, p // k, p // 2, p - p // k):
            sizes.add(p + d)
        p *= k
    return sorted(n for n in sizes if b < n <= top)


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("layout,b", [("bst", 1), ("btree", 1), ("btree", 2), ("btree", 7),
                                      ("btree", 16), ("btree", 63), ("btree", 300)])
def test_slide_emulated(emulator, layout, b, width):
    sizes = edges(b, 6000 if width == 8 else 4500)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", EMU_B=str(b))
    r = subprocess.run([emulator, layout, str(width)] + [str(n) for n in sizes],
                       capture_output=True, text=True, timeout=900, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stderr.count("0 wrong, inverse 0 wrong") == len(sizes), r.stderr[-4000:]
