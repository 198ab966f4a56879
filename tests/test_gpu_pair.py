"""Runs of steps that take two steps a pass against the same steps taken one
call at a time (which are checked against the oracle elsewhere): every core
cell, and on closed lattices every padding cell too, bit for bit in FP32, BF16
and FP64 storage (in FP16 to the last bit: a conversion may fuse with an FMA in
one kernel and not in the other, which a few steps carry on), at extents that
are no multiple of any tile, with padding 1 to 3, with run lengths that leave
single steps over, and with statistics."""
import numpy as np
import pytest

from openlb_amd import (BGK, BOUNCE_BACK, BOUNCE_BACK_VELOCITY, FIELD_FORCE, FORCED_BGK, FORCED_TRT, NO_DYNAMICS,
                        SMAGORINSKY_BGK, TRT, Dynamics, Lattice)

pytestmark = pytest.mark.gpu

# the extents are just above the sizes from which a run takes two steps a pass
UNIFORM = [
    ("f32", BGK, (39, 41, 43), 3),       # 512 threads, one short row a tile
    ("f32", BGK, (20, 9, 513), 1),       # thin along y, long rows
    ("f32", BGK, (5, 700, 40), 2),
    ("f32", BGK, (135, 139, 131), 1),    # 1024 threads
    ("f32", FORCED_TRT, (150, 163, 149), 2),
    ("f32", SMAGORINSKY_BGK, (161, 157, 141), 3),
    ("f16", BGK, (187, 190, 201), 1),
    ("bf16", BGK, (187, 190, 201), 2),
    ("bf16", SMAGORINSKY_BGK, (201, 187, 190), 3),
    ("f64", BGK, (65, 71, 69), 3),
    ("f64", TRT, (120, 123, 122), 1),    # a uniform kind that runs masked
]
MASKED = [
    ("f32", True, (147, 155, 151), 1), ("f32", False, (151, 147, 155), 3), ("f32", False, (150, 152, 161), 1),
    ("f64", True, (119, 121, 127), 2), ("f64", False, (117, 121, 125), 1),
]


def _compare(a, b, storage, everywhere):
    fa, fb = a.get_populations(), b.get_populations()
    np.testing.assert_array_equal(a.ring_shifts(), b.ring_shifts())
    if not everywhere:
        p = a.padding
        core = np.zeros(a.shape, dtype=bool)
        core[p:-p, p:-p, p:-p] = True
        fa, fb = fa[:, core.reshape(-1)], fb[:, core.reshape(-1)]
    assert np.isfinite(fb).all()
    if storage == "f16":
        # one rounding against two of a value below 2^-6: one unit of 2^-17 a
        # step at most, carried on by a relaxation that does not amplify
        assert np.abs(fa - fb).max() <= 10 * 2.0 ** -17
    else:
        np.testing.assert_array_equal(fa, fb)


def _pair(extent, padding, periodic, storage, mask, slots, force=None):
    rng = np.random.default_rng(3)
    lats = []
    f = None
    for _ in range(2):
        lat = Lattice(extent, padding, (periodic,) * 3, storage)
        for k, d in slots.items():
            lat.set_dynamics(k, d)
        lat.set_dynamics_mask(mask)
        if force is not None:
            lat.set_cell_field(FIELD_FORCE, force)
        if f is None:
            f = (0.002 * rng.standard_normal((19, lat.ncells), dtype=np.float32)).astype(lat._dtype)
        lat.set_populations(f)
        lats.append(lat)
    return lats


def _padded(extent, padding):
    return tuple(n + 2 * padding for n in extent)


@pytest.mark.parametrize("storage,kind,extent,padding", UNIFORM)
def test_uniform_runs(storage, kind, extent, padding):
    print(f"[pair] uniform {storage} kind={kind} {extent} p{padding}", flush=True)
    mask = np.zeros(_padded(extent, padding), dtype=np.uint8)
    mask[padding:-padding, padding:-padding, padding:-padding] = 1
    dyn = Dynamics(kind, omega=1 / 0.7, magic=3 / 16, force=(1e-4, -2e-4, 5e-5), smagorinsky=0.1)
    a, b = _pair(extent, padding, True, storage, mask, {1: dyn})
    a.collide_and_stream(6)
    a.set_statistics(True)
    a.collide_and_stream(5)
    for _ in range(10):
        b.collide_and_stream(1)
    b.set_statistics(True)
    b.collide_and_stream(1)
    _compare(a, b, storage, False)
    sa, sb = a.get_statistics(), b.get_statistics()
    if storage != "f16":
        assert sa == sb
    a.close()
    b.close()


@pytest.mark.parametrize("storage,periodic,extent,padding", MASKED)
def test_masked_runs(storage, periodic, extent, padding):
    """a random mix of dynamics, a per-cell force, NoDynamics cells"""
    print(f"[pair] masked {storage} periodic={periodic} {extent} p{padding}", flush=True)
    rng = np.random.default_rng(11)
    slots = {1: Dynamics(BGK, omega=1 / 0.61), 2: Dynamics(TRT, omega=1 / 0.8, magic=0.25), 3: Dynamics(BOUNCE_BACK),
             4: Dynamics(NO_DYNAMICS), 5: Dynamics(FORCED_BGK, omega=1 / 0.7),
             6: Dynamics(BOUNCE_BACK_VELOCITY, wall_velocity=(0.02, 0.0, -0.01)),
             7: Dynamics(SMAGORINSKY_BGK, omega=1 / 0.55, smagorinsky=0.12), 8: Dynamics(FORCED_TRT, omega=1.2, magic=0.2)}
    # ids in the padding too: its cells never collide
    mask = rng.integers(1, 9, _padded(extent, padding), dtype=np.uint8)
    force = 1e-4 * rng.standard_normal((mask.size, 3))
    a, b = _pair(extent, padding, periodic, storage, mask, slots, force)
    a.collide_and_stream(9)
    for _ in range(9):
        b.collide_and_stream(1)
    _compare(a, b, storage, not periodic)
    a.close()
    b.close()


@pytest.mark.parametrize("storage,periodic,extent,padding", MASKED)
def test_bgk_with_bounce_back_runs(storage, periodic, extent, padding):
    """two BGK slots, bounce-back, a moving wall and NoDynamics cells: the
    kernel with one bulk kind"""
    print(f"[pair] walls {storage} periodic={periodic} {extent} p{padding}", flush=True)
    rng = np.random.default_rng(12)
    slots = {1: Dynamics(BGK, omega=1 / 0.61), 2: Dynamics(BGK, omega=1 / 0.9), 3: Dynamics(BOUNCE_BACK),
             4: Dynamics(NO_DYNAMICS), 6: Dynamics(BOUNCE_BACK_VELOCITY, wall_velocity=(0.02, 0.0, -0.01))}
    mask = rng.choice(np.array([1, 1, 1, 2, 3, 4, 6], dtype=np.uint8), _padded(extent, padding))
    a, b = _pair(extent, padding, periodic, storage, mask, slots)
    a.collide_and_stream(8)
    for _ in range(8):
        b.collide_and_stream(1)
    _compare(a, b, storage, not periodic)
    a.close()
    b.close()


def test_lattice_of_an_ensemble_keeps_its_buffer():
    """a member that runs on its own between ensemble steps"""
    from openlb_amd import Ensemble

    extent = (40, 41, 42)
    mask = np.zeros(_padded(extent, 1), dtype=np.uint8)
    mask[1:-1, 1:-1, 1:-1] = 1
    a, b = _pair(extent, 1, True, "f32", mask, {1: Dynamics(BGK, omega=1 / 0.6)})
    ens = Ensemble([a])
    ens.step(2)
    a.collide_and_stream(8)
    ens.step(1)
    a.collide_and_stream(4)
    a.reduce_moments()
    ens.step(2)
    for _ in range(17):
        b.collide_and_stream(1)
    _compare(a, b, "f32", False)
    ens.close()
