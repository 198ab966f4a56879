"""Moment sums over one block of partials, exactly one chunk of them, one more,
and several chunks: against the FP64 sums of the populations."""
import numpy as np
import pytest

from openlb_amd import BGK, Dynamics, Lattice
from tests.helpers import C

pytestmark = pytest.mark.gpu

# 256 cells a block, 1024 blocks a chunk: 1 block, 1024, 1025, 2 chunks and a remainder
EXTENTS = [(3, 5, 7), (32, 64, 128), (16, 128, 128 + 1), (67, 83, 101)]


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("extent", EXTENTS)
def test_moment_sums(extent, storage):
    print(f"[moments] {extent} {storage}", flush=True)
    rng = np.random.default_rng(5)
    lat = Lattice(extent, 1, (True, True, True), storage)
    mask = np.zeros(lat.shape, dtype=np.uint8)
    mask[1:-1, 1:-1, 1:-1] = rng.random(extent) < 0.9
    f = (0.002 * rng.standard_normal((19, lat.ncells), dtype=np.float32)).astype(lat._dtype)
    lat.set_dynamics(1, Dynamics(BGK, omega=1 / 0.7))
    lat.set_dynamics_mask(mask)
    lat.set_populations(f)
    got, again = lat.reduce_moments(), lat.reduce_moments()
    assert got == again
    v = f[:, mask.reshape(-1) == 1].astype(np.float64)
    j = C.T.astype(np.float64) @ v
    rho = 1 + v.sum(axis=0)
    usqr = (j**2).sum(axis=0) / rho**2
    n = v.shape[1]
    # both sides add n (or 19 n) FP64 numbers, in some order
    eps = 2.0**-52 * (n + 32)
    want = {"nCells": (n, 0), "mass": (v.sum(), eps * np.abs(v).sum()),
            "sumUSqr": (usqr.sum(), eps * usqr.sum()), "maxUSqr": (usqr.max(), 64 * 2.0**-52 * usqr.max())}
    for k, (w, tol) in want.items():
        assert abs(got[k] - w) <= tol, (k, got[k], w, tol)
    for k in range(3):
        assert abs(got["momentum"][k] - j[k].sum()) <= eps * np.abs(v).sum()
