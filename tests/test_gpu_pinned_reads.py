"""Reads into arrays that the runtime knows (pinned host memory) and into
ordinary ones: the same values, and the pinned ones, which the device writes
without a detour, the faster."""
import ctypes
import time

import numpy as np
import pytest
import torch

from openlb_amd import BGK, Dynamics, Lattice, library

pytestmark = pytest.mark.gpu


def _lattice(n):
    lat = Lattice((n, n, n), 1, (True,) * 3, "f32")
    lat.set_dynamics(1, Dynamics(BGK, omega=1 / 0.7))
    lat.set_dynamics_mask(np.ones(lat.shape, dtype=np.uint8))
    rng = np.random.default_rng(4)
    lat.set_populations(0.002 * rng.standard_normal((19, lat.ncells), dtype=np.float32))
    return lat


def test_pinned_arrays():
    print("[pinned reads] 140", flush=True)
    lat = _lattice(140)

    def arrays(pinned):
        return [torch.zeros(k * lat.ncells, dtype=torch.float32, pin_memory=pinned) for k in (1, 3)]

    def read(dst):
        assert library().olbgfx_compute_rho_u(lat._h, lat._value, *(ctypes.c_void_p(t.data_ptr()) for t in dst)) == 0

    pinned, plain = arrays(True), arrays(False)
    best = [np.inf, np.inf]
    for _ in range(8):
        for k, dst in enumerate((pinned, plain)):
            t = time.perf_counter()
            read(dst)
            best[k] = min(best[k], time.perf_counter() - t)
    for a, b in zip(pinned, plain):
        assert torch.equal(a, b)
    f = torch.zeros((19, lat.ncells), dtype=torch.float32, pin_memory=True)
    assert library().olbgfx_get_populations(lat._h, lat._value, ctypes.c_void_p(f.data_ptr())) == 0
    assert np.array_equal(f.numpy(), lat.get_populations())
    lat.close()
    # 0.93 against 1.47 ms; both took 1.47 when pinned arrays went through the ring
    assert best[0] <= 0.85 * best[1]
