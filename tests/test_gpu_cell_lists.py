"""Cell lists of every length around a workgroup, in any order, gathered and
scattered against the populations the lattice hands out: exact, in every
storage type."""
import numpy as np
import pytest
import torch  # before the library, so that both use one HIP runtime

from openlb_amd import Lattice

pytestmark = pytest.mark.gpu

WORD = {"f32": np.uint32, "f16": np.uint16, "bf16": np.uint16, "f64": np.uint64}


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 1000])
@pytest.mark.parametrize("storage", ["f32", "f16", "bf16", "f64"])
def test_gather_and_scatter(storage, n):
    print(f"[cells] {storage} n={n}", flush=True)
    rng = np.random.default_rng(n)
    a, b = (Lattice((9, 8, 11), 2, (True, False, True), storage) for _ in range(2))
    a.set_populations(rng.standard_normal((19, a.ncells)).astype(a._dtype))
    a.collide_and_stream(3)  # ring offsets that differ from population to population
    b.collide_and_stream(7)
    ids = rng.permutation(a.ncells)[:n]
    la, lb = a.cell_list(ids), b.cell_list(ids)
    buf = torch.zeros(la.nbytes, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    a.gather_cells(la, buf.data_ptr(), stream)
    b.scatter_cells(lb, buf.data_ptr(), stream)
    torch.cuda.synchronize()
    fa, fb = a.get_populations(), b.get_populations()
    np.testing.assert_array_equal(fb[:, ids], fa[:, ids])
    others = np.setdiff1d(np.arange(a.ncells), ids)
    assert not fb[:, others].any()
    words = buf.cpu().numpy().view(WORD[storage]).reshape(19, n)
    if storage == "f32":
        np.testing.assert_array_equal(words.view(np.float32), fa[:, ids])
    if storage == "f64":
        np.testing.assert_array_equal(words.view(np.float64), fa[:, ids])
