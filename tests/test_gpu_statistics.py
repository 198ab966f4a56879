"""Lattice statistics of lattices whose blocks fill one reduction block, just
more than one, and many: against the FP64 sums of the same step's
populations, and independent of how many steps a call takes."""
import numpy as np
import pytest

from openlb_amd import BGK, Dynamics, Lattice
from tests.helpers import C

pytestmark = pytest.mark.gpu

# 256 cells a block: 1 block, 2048 blocks, 2049, and several chunks of 2048
EXTENTS = [(4, 8, 8), (32, 128, 128), (32, 128, 128 + 1), (160, 121, 131)]


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("extent", EXTENTS)
def test_statistics_of_the_last_step(extent, storage):
    print(f"[stats] {extent} {storage}", flush=True)
    rng = np.random.default_rng(2)
    one, run = (Lattice(extent, 1, (True, True, True), storage) for _ in range(2))
    mask = np.zeros(one.shape, dtype=np.uint8)
    mask[1:-1, 1:-1, 1:-1] = 1
    f = (0.002 * rng.standard_normal((19, one.ncells), dtype=np.float32)).astype(one._dtype)
    for lat in (one, run):
        lat.set_dynamics(1, Dynamics(BGK, omega=1 / 0.7))
        lat.set_dynamics_mask(mask)
        lat.set_populations(f)
        lat.set_statistics(True)
    for _ in range(2):
        one.collide_and_stream(1)
    before = one.get_populations()[:, mask.reshape(-1) == 1].astype(np.float64)
    one.collide_and_stream(1)
    run.collide_and_stream(3)
    a, b = one.get_statistics(), run.get_statistics()
    assert a == b
    # the third step's statistics are the moments of the populations it collides
    rho = 1 + before.sum(axis=0)
    usqr = ((C.T.astype(np.float64) @ before / rho) ** 2).sum(axis=0)
    # FP32 moments: 19 terms of 2^-24 relative to the largest partial sum, about
    # 0.02, in rho, and three times that in u^2
    tol = 1e-12 if storage == "f64" else 1e-6
    assert a["nCells"] == np.prod(extent)
    assert abs(a["sumRho"] - rho.sum()) <= tol * rho.sum()
    assert abs(a["sumUSqr"] - usqr.sum()) <= 3 * tol * usqr.sum()
    assert abs(a["maxU"] ** 2 - usqr.max()) <= 10 * tol * usqr.max()
