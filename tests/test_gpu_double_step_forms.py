"""Every form of the kernel that takes two steps a pass, against the same steps
taken singly, bit for bit, and with a look at how many steps went in pairs, so
that no row can pass by comparing single steps with themselves.  Runs of 14
steps, and of 13 with statistics, take 12 in pairs: rings to flat, flat to flat
four times and flat to rings.  Also the layout of planes too large for rows side
by side, a captured run, and a run that the memory limit refuses."""
import numpy as np
import pytest
import torch  # before the library, so that both use one HIP runtime

from openlb_amd import (BGK, BOUNCE_BACK, BOUNCE_BACK_VELOCITY, FIELD_FORCE, FORCED_BGK, FORCED_TRT, NO_DYNAMICS,
                        SMAGORINSKY_BGK, TRT, Dynamics, Lattice)

pytestmark = pytest.mark.gpu

UNIFORM = {"bgk": Dynamics(BGK, omega=1 / 0.6), "smagorinsky": Dynamics(SMAGORINSKY_BGK, omega=1 / 0.55, smagorinsky=0.12),
           "trt": Dynamics(TRT, omega=1 / 0.8, magic=0.25),
           "forced_trt": Dynamics(FORCED_TRT, omega=1.3, magic=0.2, force=(1e-4, 0.0, -2e-5))}
WALLS = {1: UNIFORM["bgk"], 2: Dynamics(BGK, omega=1 / 0.9), 3: Dynamics(BOUNCE_BACK), 4: Dynamics(NO_DYNAMICS),
         6: Dynamics(BOUNCE_BACK_VELOCITY, wall_velocity=(0.02, 0.0, -0.01))}
MIXED = {**WALLS, 2: UNIFORM["trt"], 5: Dynamics(FORCED_BGK, omega=1 / 0.7), 7: UNIFORM["smagorinsky"],
         8: UNIFORM["forced_trt"]}

FORMS = [
    ("f32", "bgk", True, (41, 44, 46), 1),        # 512 threads, one plane a tile
    ("f32", "bgk", True, (66, 68, 62), 3),        # several planes
    ("f32", "bgk", True, (150, 163, 149), 2),     # 1024 threads
    ("f32", "forced_trt", True, (150, 163, 149), 2),
    ("f32", "smagorinsky", True, (161, 157, 141), 3),
    ("f32", "trt", True, (150, 163, 149), 1),     # a uniform kind that runs masked
    ("f32", "walls", True, (150, 163, 149), 1),
    ("f32", "walls", False, (151, 157, 155), 3),
    ("f32", "mixed", True, (150, 163, 149), 1),
    ("f32", "mixed", False, (150, 162, 161), 1),
    ("f16", "bgk", True, (221, 223, 224), 1),     # 1024 threads; 512 in test_gpu_double_steps
    ("f16", "forced_trt", True, (187, 190, 201), 2),
    ("bf16", "bgk", True, (187, 190, 201), 2),    # 512 threads
    ("bf16", "forced_trt", True, (344, 250, 86), 1),
    ("f64", "bgk", True, (65, 71, 69), 3),
    ("f64", "bgk", True, (133, 134, 137), 1),
    ("f64", "forced_trt", True, (131, 139, 142), 1),
    ("f64", "smagorinsky", True, (133, 134, 137), 2),
    ("f64", "trt", True, (131, 139, 142), 1),
    ("f64", "walls", True, (133, 134, 137), 1),
    ("f64", "walls", False, (131, 139, 142), 1),
    ("f64", "mixed", True, (133, 134, 137), 2),
    ("f64", "mixed", False, (131, 139, 142), 1),
]


def _lattice(storage, kind, periodic, extent, padding, seed=11):
    rng = np.random.default_rng(seed)
    lat = Lattice(extent, padding, (periodic,) * 3, storage)
    slots = {"walls": WALLS, "mixed": MIXED}.get(kind) or {1: UNIFORM[kind]}
    for k, d in slots.items():
        lat.set_dynamics(k, d)
    if kind in UNIFORM:
        mask = np.zeros(lat.shape, dtype=np.uint8)
        mask[tuple(slice(padding, -padding) for _ in range(3))] = 1
    else:
        # ids in the padding too: its cells never collide
        mask = rng.choice(np.array([1, 1, *slots], dtype=np.uint8), lat.shape)
    lat.set_dynamics_mask(mask)
    if kind == "mixed":
        lat.set_cell_field(FIELD_FORCE, 1e-4 * rng.standard_normal((lat.ncells, 3)))
    lat.set_populations((0.002 * rng.standard_normal((19, lat.ncells), dtype=np.float32)).astype(lat._dtype))
    return lat


def _assert_equal(a, b, everywhere):
    fa, fb = a.get_populations(), b.get_populations()
    np.testing.assert_array_equal(a.ring_shifts(), b.ring_shifts())
    if not everywhere:
        core = np.zeros(a.shape, dtype=bool)
        core[tuple(slice(a.padding, -a.padding) for _ in range(3))] = True
        fa, fb = fa[:, core.reshape(-1)], fb[:, core.reshape(-1)]
    assert np.isfinite(fb).all()
    np.testing.assert_array_equal(fa, fb)


@pytest.mark.parametrize("storage,kind,periodic,extent,padding", FORMS)
def test_forms(storage, kind, periodic, extent, padding):
    print(f"[double step forms] {storage} {kind} periodic={periodic} {extent} p{padding}", flush=True)
    a, b = (_lattice(storage, kind, periodic, extent, padding) for _ in range(2))
    b.set_two_step(0)
    a.collide_and_stream(14)
    b.collide_and_stream(14)
    assert a.get_two_step()[1] == 12 and b.get_two_step() == (0, 0)
    _assert_equal(a, b, not periodic)
    for lat in (a, b):
        lat.set_statistics(True)
        lat.collide_and_stream(13)
    assert a.get_two_step()[1] == 24
    assert a.get_statistics() == b.get_statistics()
    _assert_equal(a, b, not periodic)
    a.close()
    b.close()


def test_captured_run_takes_single_steps():
    print("[double step forms] capture", flush=True)
    a, b, c = (_lattice("f32", "bgk", True, (66, 68, 62), 2) for _ in range(3))
    c.set_two_step(0)
    stream = torch.cuda.Stream()
    for lat in (a, b, c):
        lat.collide_and_stream(8, stream.cuda_stream)
    stream.synchronize()
    assert a.get_two_step()[1] == 8
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        a.collide_and_stream(9, stream.cuda_stream)
    assert a.get_two_step()[1] == 8
    graph.replay()
    torch.cuda.synchronize()
    b.collide_and_stream(9)
    c.collide_and_stream(9)
    assert b.get_two_step()[1] == 16
    _assert_equal(a, c, False)
    _assert_equal(b, c, False)
    a.collide_and_stream(8)  # and the lattice goes on from there
    c.collide_and_stream(8)
    assert a.get_two_step()[1] == 16
    _assert_equal(a, c, False)
    for lat in (a, b, c):
        lat.close()


def test_large_planes():
    """rows side by side would put a plane's offsets beyond 32 bits"""
    extent = (4, 5400, 5400)
    print(f"[double step forms] f64 bgk {extent}", flush=True)
    mask = np.zeros(tuple(n + 2 for n in extent), dtype=np.uint8)
    mask[1:-1, 1:-1, 1:-1] = 1
    ids = np.flatnonzero(mask.reshape(-1)).astype(np.uint32)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    start = torch.empty((19, ids.size), dtype=torch.float64, device="cuda").normal_(0.0, 0.002, generator=gen)
    out = torch.empty_like(start)
    torch.cuda.synchronize()
    for pairs in (True, False):
        lat = Lattice(extent, 1, (True,) * 3, "f64")
        lat.set_dynamics(1, UNIFORM["bgk"])
        lat.set_dynamics_mask(mask)
        if not pairs:
            lat.set_two_step(0)
        cells = lat.cell_list(ids)
        lat.scatter_cells(cells, start.data_ptr())
        lat.collide_and_stream(9)
        assert lat.get_two_step()[1] == (8 if pairs else 0)
        # the single steps' result takes the place of the inputs
        lat.gather_cells(cells, (out if pairs else start).data_ptr())
        lat.synchronize()
        cells.close()
        lat.close()
    assert torch.equal(out, start)
    del out, start
    torch.cuda.empty_cache()
