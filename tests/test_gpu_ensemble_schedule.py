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


@pytest.mark.parametrize("group_bytes,per_group,ticket", [(0, 1, False), (1 << 20, 33, False), (1 << 20, 4, True)])
def test_offsets_of_many_steps(group_bytes, per_group, ticket):
    """32 steps' offsets are formed at once: calls of 31, 32, 33 and 65 steps,
    on edges so short that the offsets wrap within them"""
    print(f"[ensemble schedule] offsets {group_bytes} {per_group} {ticket}", flush=True)
    lats = ([], [])
    for k, n in enumerate((3, 9, 24, 17)):
        case = cases.box_cavity(n, u_lid=0.03 + 0.01 * k, dtype=np.float32)
        for group in lats:
            lat = Lattice(case.extent, case.padding, case.periodic, "f32")
            case.apply(lat)
            group.append(lat)
    ens = Ensemble(lats[0])
    if per_group > 1:
        ens.set_schedule(group_bytes, per_group, ticket)
    for steps in (31, 32, 33, 65):
        ens.step(steps)
    ens.capture(33)
    ens.launch_graph(2)
    for a, b in zip(*lats):
        for _ in range(227):
            b.collide_and_stream(1)
        np.testing.assert_array_equal(a.ring_shifts(), b.ring_shifts())
        np.testing.assert_array_equal(a.get_populations(), b.get_populations())
