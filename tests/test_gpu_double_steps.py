"""Runs that take two steps a pass: in 2-byte storage against the same steps one
a call, bit for bit (a conversion to FP16 that fuses with the last FMA of a
collision in one kernel has to fuse in the other too), and what they do with
memory.  Runs of 14 steps go through all three passes (rings to flat, flat to
flat, flat to rings)."""
import threading

import numpy as np
import pytest
import torch

from openlb_amd import BGK, FORCED_TRT, Dynamics, Lattice, cases

pytestmark = pytest.mark.gpu

KINDS = {"bgk": Dynamics(BGK, omega=1 / 0.6), "forced_trt": Dynamics(FORCED_TRT, omega=1.3, magic=0.2,
                                                                     force=(1e-4, 0.0, -2e-5))}


def _core(extent, padding):
    mask = np.zeros(tuple(n + 2 * padding for n in extent), dtype=np.uint8)
    mask[padding:-padding, padding:-padding, padding:-padding] = 1
    return mask


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("extent", [(187, 190, 201), (1030, 257, 258)], ids=["7M", "68M"])
def test_two_byte_runs(extent, storage, kind):
    """both workgroup sizes: 1024 threads, and 512 from 64 M cells"""
    print(f"[double steps] {storage} {kind} {extent}", flush=True)
    mask = _core(extent, 1)
    ids = np.flatnonzero(mask.reshape(-1)).astype(np.uint32)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16}[storage]
    start = torch.empty((19, ids.size), dtype=dtype, device="cuda").normal_(0.0, 0.002, generator=gen)
    torch.cuda.synchronize()
    out = []
    for calls in ([14, 5], [1] * 19):
        lat = Lattice(extent, 1, (True,) * 3, storage)
        lat.set_dynamics(1, KINDS[kind])
        lat.set_dynamics_mask(mask)
        cells = lat.cell_list(ids)
        lat.scatter_cells(cells, start.data_ptr())
        for steps in calls:
            lat.collide_and_stream(steps)
        got = torch.empty_like(start)
        lat.gather_cells(cells, got.data_ptr())
        lat.synchronize()
        out.append(got.view(torch.int16))
        cells.close()
        lat.close()
    assert torch.equal(out[0], out[1])


def _tgv(n):
    case = cases.tgv(n, dtype=np.float32)
    lat = Lattice(case.extent, case.padding, case.periodic, "f32")
    case.apply(lat)
    return case, lat


def test_second_set_is_limited_and_given_back():
    print("[double steps] memory", flush=True)
    case, lat = _tgv(160)
    _, single = _tgv(160)
    single.set_two_step(0)
    size = 19 * 4 * lat.ncells
    free = torch.cuda.mem_get_info()[0]
    lat.collide_and_stream(8)
    held, steps = lat.get_two_step()
    assert held >= size and steps == 8
    lat.synchronize()
    assert torch.cuda.mem_get_info()[0] <= free - size
    lat.set_two_step(held)                      # fits: kept
    assert lat.get_two_step() == (held, 8)
    lat.set_two_step(held - 1)                  # given back, and not taken again
    assert lat.get_two_step() == (0, 8)
    assert torch.cuda.mem_get_info()[0] >= free - size // 8
    lat.collide_and_stream(6)
    assert lat.get_two_step() == (0, 8)
    lat.set_two_step()
    lat.collide_and_stream(7)
    assert lat.get_two_step() == (held, 12)
    single.collide_and_stream(21)
    assert single.get_two_step() == (0, 0)
    core = case.core_mask().reshape(-1)
    np.testing.assert_array_equal(lat.get_populations()[:, core], single.get_populations()[:, core])
    lat.close()
    single.close()


def test_first_run_leaves_a_capture_of_another_thread_alone():
    """the first run of a lattice allocates; a stream that another thread is
    capturing must not notice"""
    print("[double steps] another thread captures", flush=True)
    case, lat = _tgv(64)
    _, ref = _tgv(64)
    ref.collide_and_stream(8)
    ref.synchronize()
    side, own = torch.cuda.Stream(), torch.cuda.Stream()
    x = torch.zeros(256, device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    errors = []

    def run():
        try:
            lat.collide_and_stream(8, own.cuda_stream)
        except Exception as exc:
            errors.append(exc)

    with torch.cuda.graph(graph, stream=side, capture_error_mode="global"):
        x.add_(1.0)
        thread = threading.Thread(target=run)
        thread.start()
        thread.join()
        x.add_(1.0)
    assert not errors
    own.synchronize()
    x.zero_()
    for k in (1, 2, 3):
        graph.replay()
        torch.cuda.synchronize()
        assert x.tolist() == [2.0 * k] * 256
    assert lat.get_two_step()[1] == 8
    core = case.core_mask().reshape(-1)
    np.testing.assert_array_equal(lat.get_populations()[:, core], ref.get_populations()[:, core])
    lat.close()
    ref.close()
