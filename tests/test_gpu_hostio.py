"""Host copies of parcels, tendencies and fields: chunked staging against what
was stored, at the sizes where chunks, units and threads end.

What goes up comes back exactly (values representable in FP32; positions
FP64), whatever order the slots are in."""
import numpy as np
import pytest

from epic_amd import workloads as W
from epic_amd.core import FIELDS, Member

pytestmark = pytest.mark.gpu


def _f32(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32).astype(np.float64)


# the staging buffers hold 493,446 parcels: one chunk, one over, several
@pytest.mark.parametrize("n", [0, 1, 3, 1000, 493446, 493447, 1234567])
def test_parcels_round_trip(n):
    print(f"host copies: {n} parcels", flush=True)
    rng = np.random.default_rng(n)
    gm = Member(16, 12, 10, (0.0, 0.0, 0.0), (1.0, 0.75, 0.625), max_parcels=n + 5)
    pos = rng.uniform(0.0, 1.0, (n, 3)) * (1.0, 0.75, 0.625)
    want = {"position": pos, "vorticity": _f32(rng, n, 3), "B": _f32(rng, n, 5), "volume": _f32(rng, n),
            "buoyancy": _f32(rng, n), "humidity": _f32(rng, n)}
    gm.set_parcels(*want.values())
    got = gm.get_parcels()
    for k, v in want.items():
        assert np.array_equal(got[k], v), k
    gm.resort()   # the slots in cell order, the caller's order as before
    dp, dv = _f32(rng, n, 3), _f32(rng, n, 3)
    gm.set_tendencies(dp, dv)
    got = gm.get_parcels()
    for k, v in want.items():
        assert np.array_equal(got[k], v), k
    gp, gv, st = gm.get_tendencies()
    assert np.array_equal(gp, dp) and np.array_equal(gv, dv) and st.shape == (n, 8)


# units of 32 x columns, tiles of 32 z: below, at and above both
@pytest.mark.parametrize("grid", [(8, 8, 4), (30, 9, 30), (32, 8, 27), (64, 10, 64), (96, 128, 80)])
def test_fields_round_trip(grid):
    nx, ny, nz = grid
    print(f"host copies: fields of {grid}", flush=True)
    gm = Member(nx, ny, nz, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
    rng = np.random.default_rng(5)
    for name in ("volg", "velgradg"):
        nc = FIELDS[name][1]
        f = _f32(rng, nc, nx + 3, ny + 3, nz + 3)
        gm.set_field(name, f)
        got = gm.get_field(name).reshape(f.shape)
        # the interior columns come back, and the x and y halos are periodic
        ix, iy = (np.arange(-1, nx + 2) % nx) + 1, (np.arange(-1, ny + 2) % ny) + 1
        assert np.array_equal(got, f[:, ix][:, :, iy])


def test_counts_as_both_types():
    mem = W.rising_thermal(16, seed=3)
    gm = Member.from_workload(mem)
    gm.par2grid()
    a = gm.get_field("nparg")
    assert a.dtype == np.int32 and a[1:17, 1:17].sum() == mem.n
