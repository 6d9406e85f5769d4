"""The emulator's Makefile: a header that several programs include is written
by a rule of its own, and every program that includes it waits for it (two
rules that write one file empty it for each other under make -j)."""
import os
import re
import subprocess

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


def test_small_partition_header_has_one_writer():
    db = subprocess.run(["make", "-C", EMU, "-npq", "all"], capture_output=True, text=True).stdout
    header = "_build/src/small_partition.hpp"
    rules = dict(re.findall(r"^(_build/\S+): (.*)$", db, re.M))
    assert header in rules
    for user in ("src/tl_part.cpp", "src/tl_sort2.cpp", "emu_part", "emu_sort2"):
        assert header in rules["_build/" + user].split(), user
    makefile = open(os.path.join(EMU, "Makefile")).read()
    assert not re.search(r">\s*\S*small_partition\.hpp", makefile)
