"""Field copies on every route: as they lie on the device (up to 160 KB down and
320 KB up, planes not whole pages apart, more than 16 KB down), by a launch on
the pinned memory itself, and in chunks that end within a component."""
import numpy as np
import pytest

from epic_amd.core import FIELDS, Member

pytestmark = pytest.mark.gpu

GRIDS = [
    (8, 9, 4),        # the smallest: as they lie up, on pinned memory down
    (16, 32, 5),      # 16 KB a component
    (16, 32, 6),      # and more
    (30, 9, 30),      # 3 components below 160 KB, 8 between that and 320 KB
    (20, 32, 64),     # one component just above 160 KB, three above 320
    (32, 32, 16),     # whole pages: pinned memory, and a copy for 8 components
    (40, 40, 125),    # z blocks with a remainder, columns not a multiple of 32
    (128, 128, 80),   # 44 MB: two chunks
]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_round_trip(grid):
    nx, ny, nz = grid
    print(f"field copies: {grid}", flush=True)
    gm = Member(nx, ny, nz, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
    rng = np.random.default_rng(nx + ny + nz)
    ix, iy = (np.arange(-1, nx + 2) % nx) + 1, (np.arange(-1, ny + 2) % ny) + 1
    kept = {}
    for name in ("volg", "velog", "velgradg", "vtend"):
        f = rng.standard_normal((FIELDS[name][1], nx + 3, ny + 3, nz + 3)).astype(np.float32).astype(np.float64)
        gm.set_field(name, f)
        kept[name] = f[:, ix][:, :, iy]   # the interior columns, and periodic halos
    for name, want in kept.items():   # no upload touched another field
        assert np.array_equal(gm.get_field(name).reshape(want.shape), want), name
