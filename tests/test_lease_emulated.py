"""The query workspaces' leases on the CPU (tests/emu/emu_lease.cpp): a call whose
workspace grows holds no other call up, somewhat larger batches need no new
memory, idle workspaces can be given back, short memory is no error."""
import os
import subprocess

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


def test_leases():
    subprocess.run(["make", "-C", EMU, "-j4", "_build/emu_lease"], check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([os.path.join(EMU, "_build", "emu_lease")], capture_output=True, text=True,
                       timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
    assert r.stdout.count(": right") == 12, r.stdout
