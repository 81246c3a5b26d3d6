"""Staging buffers of the host copies, seen from the allocator (a child process
whose large allocations pass through alloc_watch.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
watch = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
import numpy as np
from epic_amd import workloads as W
from epic_amd.core import Member
refuse = C.c_int.in_dll(watch, "watch_refuse_device")
device, pinned = (C.c_long.in_dll(watch, n) for n in ("watch_device", "watch_pinned"))
"""


def _run(tmp_path, body):
    lib = str(tmp_path / "alloc_watch.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "alloc_watch.cpp"), "-ldl"], check=True)
    code = PRELUDE.format(root=os.path.dirname(HERE), lib=lib) + body
    print("staging: child process", flush=True)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_one_set_stays_when_the_last_member_goes(tmp_path):
    _run(tmp_path, """
def cycle():
    mem = W.rising_thermal(32, seed=3)
    gm = Member.from_workload(mem)
    gm.par2grid()
    gm.get_field("velgradg"), gm.get_tendencies(), gm.get_parcels()
    gm.close()
    return pinned.value

first = cycle()
assert first > 0, "the allocator is not watched"
assert cycle() == first, "pinned buffers allocated again for the next member"
""")


def test_copies_need_no_device_memory(tmp_path):
    _run(tmp_path, """
rng = np.random.default_rng(1)
f32 = lambda *s: rng.standard_normal(s).astype(np.float32).astype(np.float64)
grid, n = (96, 128, 80), 600001   # several chunks each
gm = Member(*grid, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), max_parcels=n)
small = Member(16, 16, 16, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
refuse.value = 1
want = [rng.uniform(0.0, 1.0, (n, 3)), f32(n, 3), f32(n, 5), f32(n), f32(n), f32(n)]
gm.set_parcels(*want)
assert all(np.array_equal(a, b) for a, b in zip(gm.get_parcels().values(), want))
dp, dv = f32(n, 3), f32(n, 3)
gm.set_tendencies(dp, dv)
got = gm.get_tendencies()
assert np.array_equal(got[0], dp) and np.array_equal(got[1], dv)
for m, g in ((gm, grid), (small, (16, 16, 16))):
    f = f32(8, *(k + 3 for k in g))
    m.set_field("velgradg", f)
    got = m.get_field("velgradg")
    assert np.array_equal(got[:, 1:-2, 1:-2], f[:, 1:-2, 1:-2])
assert device.value > 0, "the allocator is not watched"
""")


def test_idle_buffers_give_way(tmp_path):
    """An allocation that finds device memory short gets it once the idle
    staging buffers are back."""
    _run(tmp_path, """
mem = W.rising_thermal(32, seed=3)
gm = Member.from_workload(mem)
gm.get_parcels()
held = device.value
refuse.value = -1   # the launch tables of the next call
gm.par2grid()
gm.get_parcels()
assert device.value > held, "no staging buffers were given back"
""")
