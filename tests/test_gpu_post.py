"""The post-processors of velocity boundaries on boxes so small that the edges
hold less than a wave's 8 cells, just as many, and a remainder, against the
oracle: FP32 within 1e-5 of the unshifted populations, FP64 within 1e-12."""
import numpy as np
import pytest

from openlb_amd import Lattice, cases
from oracle.oracle import OracleLattice
from tests.helpers import core_cells, rel_err_unshifted

pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-5, "f64": 1e-12}


def _run(case, storage):
    lats = []
    for cls in (Lattice, OracleLattice):
        lat = cls(case.extent, case.padding, case.periodic, storage)
        case.apply(lat)
        lat.collide_and_stream(20)
        lats.append(lat)
    return lats


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("res", [4, 5, 9, 10])
def test_cavity_edges_and_corners(res, storage):
    print(f"[post] cavity res={res} {storage}", flush=True)
    case = cases.cavity3d_local_velocity(res, dtype=np.float64 if storage == "f64" else np.float32)
    gpu, orc = _run(case, storage)
    # edge and corner cells hold rewritten populations; on faces those that
    # enter from the padding are rebuilt, on fluid cells all are streamed
    edge = np.zeros(case.extent, dtype=int)
    for ax in range(3):
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[ax], hi[ax] = 0, -1
        edge[tuple(lo)] += 1
        edge[tuple(hi)] += 1
    cells = np.zeros(case.shape, dtype=bool)
    p = case.padding
    cells[p:-p, p:-p, p:-p] = edge != 1
    cells = cells.reshape(-1)
    assert rel_err_unshifted(gpu.get_populations()[:, cells], orc.get_populations()[:, cells]) <= TOL[storage]


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("ny,nz", [(3, 4), (5, 6), (10, 7), (19, 18)])
def test_interpolated_faces(ny, nz, storage):
    print(f"[post] channel {ny}x{nz} {storage}", flush=True)
    case = cases.channel3d(12, ny, nz, boundary="interpolated", dtype=np.float64 if storage == "f64" else np.float32)
    gpu, orc = _run(case, storage)
    cells = core_cells(case) & np.isin(case.materials.reshape(-1), (1, 3, 4))
    assert rel_err_unshifted(gpu.get_populations()[:, cells], orc.get_populations()[:, cells]) <= TOL[storage]
