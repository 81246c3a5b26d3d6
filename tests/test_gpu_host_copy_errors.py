"""Host copies beside failures that are not theirs: an error that another HIP
call left in the thread's last-error slot."""
import ctypes as C
import re

import numpy as np
import pytest

from epic_amd import workloads as W
from epic_amd.core import Member

pytestmark = pytest.mark.gpu


def _hip():
    """The HIP runtime that the library uses."""
    for line in open("/proc/self/maps"):
        m = re.search(r"(/opt/rocm\S*/libamdhip64\.so\S*)$", line.strip())
        if m:
            return C.CDLL(m.group(1))
    pytest.skip("no /opt/rocm HIP runtime mapped")


def test_copies_ignore_an_earlier_error():
    mem = W.rising_thermal(16, seed=3)
    gm = Member.from_workload(mem)
    gm.par2grid()
    gm.grid2par()
    hip = _hip()

    def leave_error():
        assert hip.hipSetDevice(9999) != 0   # refused on the host; nothing runs

    want = gm.get_parcels()
    leave_error()
    got = gm.get_parcels()
    for k, v in want.items():
        assert np.array_equal(got[k], v), k
    leave_error()
    f = gm.get_field("vortg")
    leave_error()
    gm.set_field("vortg", f)
    leave_error()
    dp, dv, _ = gm.get_tendencies()
    leave_error()
    gm.set_tendencies(dp, dv)
    leave_error()
    gm.set_parcels(*(want[k] for k in ("position", "vorticity", "B", "volume", "buoyancy", "humidity")))
    hip.hipGetLastError()
    got = gm.get_parcels()
    for k, v in want.items():
        assert np.array_equal(got[k], v), k
