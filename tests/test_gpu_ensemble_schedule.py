"""The default schedule of an ensemble whose members fill more than one group:
calls short enough for one launch over all groups, longer ones that advance
group after group, and a captured graph, against members stepped one by one,
bit for bit."""
import numpy as np
import pytest

from openlb_amd import Ensemble, Lattice, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,sizes", [("f32", (96, 33, 97, 101, 20, 90)), ("f16", (130, 41, 129, 128))])
def test_groups(storage, sizes):
    print(f"[ensemble schedule] {storage} {sizes}", flush=True)
    lats = ([], [])
    for k, n in enumerate(sizes):
        case = cases.box_cavity(n, u_lid=0.03 + 0.01 * k, dtype=np.float32)
        for group in lats:
            lat = Lattice(case.extent, case.padding, case.periodic, storage)
            case.apply(lat)
            group.append(lat)
    ens = Ensemble(lats[0])
    for steps in (1, 3, 4, 7):
        ens.step(steps)
    ens.capture(5)
    ens.launch_graph(2)
    for a, b in zip(*lats):
        for _ in range(25):
            b.collide_and_stream(1)
        np.testing.assert_array_equal(a.ring_shifts(), b.ring_shifts())
        np.testing.assert_array_equal(a.get_populations(), b.get_populations())
