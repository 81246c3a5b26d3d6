"""par2grid where tiles end: a last tile of a single row (the box of the tile
before it reaches over the seam), and humid air on ragged tiles and on every
launch form, against the FP64 oracle at the repository's bar (max-rel 1e-5,
counts exact)."""
import numpy as np
import pytest

from epic_amd import workloads as W
from epic_amd.core import Member
from tests._util import maxrel, oracle_state

pytestmark = pytest.mark.gpu

TOL = 1.0e-5


GRIDS = [
    (16, 25, 10, False),    # ny = 8 m + 1: row 0 lies in three boxes along y
    (16, 25, 10, True),
    (8, 25, 8, False),      # and on a grid of one tile in x
    (8, 25, 8, True),
    (16, 81, 8, False),
    (10, 225, 4, False),
    (18, 24, 10, True),     # partial tiles, 1024 threads
    (64, 40, 15, True),     # 512 threads
    (64, 64, 27, True),     # chunks of four layers
]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g[:3])) + ("-humid" if g[3] else ""))
def test_node_sums(grid):
    nx, ny, nz, humid = grid
    print(f"par2grid edges: {grid}", flush=True)
    # (ellipsoids of aspect ratio up to 4: their points reach over the seam)
    mem = W.rising_thermal(nx, seed=3 + nx + ny + nz, ny=ny, nz=nz, humidity_plume=humid, n_blobs=4 if humid else 0)
    st, gm = oracle_state(mem), Member.from_workload(mem)
    st.par2grid()
    gm.par2grid()
    sl = (Ellipsis, slice(1, nx + 1), slice(1, ny + 1), slice(None))
    for f in ("volg", "vortg", "tbuoyg", "dbuoyg", "humg"):
        assert maxrel(gm.get_field(f)[sl], getattr(st, f)[sl]) <= TOL, f
    assert np.array_equal(gm.get_field("nparg")[sl], st.nparg[sl])
    # every parcel's volume is on the grid once: planes 0 and nz hold twice
    # their share (node values are FP32, contributions 2^-28 of the largest)
    v = gm.get_field("volg")[sl][..., 1:nz + 2]
    total = v.sum() - 0.5 * (v[..., 0].sum() + v[..., nz].sum())
    assert abs(total / mem.volume.sum() - 1.0) <= 1e-6
    if ny % 2:   # (the oracle's wavenumbers are those of even lengths)
        return
    # and one step, whose stages sort and scatter what the push left
    st, gm = oracle_state(mem), Member.from_workload(mem)
    dt = 0.001
    st.ls_rk_step(0.0, dt)
    gm.ls_rk_step(0.0, dt)
    p = gm.get_parcels()
    assert np.abs(p["position"] - st.position).max() <= TOL * max(mem.dx)
    for k in ("vorticity", "B"):
        assert maxrel(p[k], getattr(st, k)) <= TOL, k


@pytest.mark.parametrize("tz", [2, 8])   # 256 and 1024 threads; 512 by default
def test_humid_tilings_give_the_same_bits(tz):
    print(f"par2grid edges: humid, chunks of {tz} layers", flush=True)
    mem = W.rising_thermal(64, seed=21, ny=72, nz=27, humidity_plume=True, n_blobs=4)
    a, b = Member.from_workload(mem), Member.from_workload(mem)
    b.set_tiling(tz, tz)
    for gm in (a, b):
        gm.ls_rk_step(0.0, 0.001)
        gm.par2grid()
    for f in ("volg", "vortg", "tbuoyg", "dbuoyg", "humg", "nparg"):
        assert np.array_equal(a.get_field(f), b.get_field(f)), f
    p, q = a.get_parcels(), b.get_parcels()
    for k in p:
        assert np.array_equal(p[k], q[k]), k
