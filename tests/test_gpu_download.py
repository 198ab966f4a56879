"""Populations, density and velocity that fill the pinned ring of the download
less than once, exactly, and several times over, from one thread and from
several."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from openlb_amd import BGK, Dynamics, Lattice

pytestmark = pytest.mark.gpu

SLOT = 2 << 20
# padded cells: 4 slots of FP32 to the byte (the least that takes the ring),
# one row under, 5 slots and a remainder, 17 of FP64 (the ring has 16)
EXTENTS = [(126, 126, 126), (126, 126, 125), (126, 126, 160), (126, 126, 268)]


def lattice(extent, storage, seed):
    rng = np.random.default_rng(seed)
    lat = Lattice(extent, 1, (True, True, True), storage)
    f = (0.002 * rng.standard_normal((19, lat.ncells), dtype=np.float32)).astype(lat._dtype)
    lat.set_dynamics(1, Dynamics(BGK, omega=1 / 0.7))
    lat.set_dynamics_mask(np.ones(lat.shape, dtype=np.uint8))
    lat.set_populations(f)
    return lat, f


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("extent", EXTENTS)
def test_download(extent, storage):
    print(f"[download] {extent} {storage}", flush=True)
    lat, f = lattice(extent, storage, 3)
    assert np.array_equal(lat.get_populations(), f)
    rho, u = lat.compute_rho_u()
    # density: 19 additions of numbers below 1.1, in the storage's precision
    eps = np.finfo(lat._dtype).eps
    want = 1 + f.sum(axis=0, dtype=np.float64)
    assert np.abs(np.asarray(rho).reshape(-1) - want).max() <= 20 * 1.1 * eps
    again = lat.compute_rho_u()
    assert np.array_equal(rho, again[0]) and np.array_equal(u, again[1])


def test_downloads_of_several_threads():
    print("[download] threads", flush=True)
    pairs = [lattice((126, 126, 130 + 3 * k), "f32", k) for k in range(3)]
    with ThreadPoolExecutor(3) as pool:
        for _ in range(2):
            got = list(pool.map(lambda p: p[0].get_populations(), pairs))
            for g, (_, f) in zip(got, pairs):
                assert np.array_equal(g, f)
    # the ring goes with the last lattice and comes back with the next
    for lat, _ in pairs:
        lat.close()
    lat, f = lattice((126, 126, 140), "f32", 9)
    assert np.array_equal(lat.get_populations(), f)
