"""What a lattice or an ensemble is launched with until a call sets it, against
the settings the library offers: the default must not be the slower one.  Times
are the least of alternating turns; the margins are half of the loss each rule
was changed for."""
import time

import numpy as np
import pytest

from openlb_amd import Lattice, cases

pytestmark = pytest.mark.gpu


def least(turns, repeats=6):
    """the least time of each turn, the turns taken one after another"""
    best = [np.inf] * len(turns)
    for _ in range(repeats):
        for k, turn in enumerate(turns):
            t = time.perf_counter()
            turn()
            best[k] = min(best[k], time.perf_counter() - t)
    return best


@pytest.mark.parametrize("res", [150, 170])
def test_velocity_boundaries_take_no_occupancy_cap(res):
    """a cap of 4 waves a SIMD costs 15 % at 150 and 10 % at 170"""
    print(f"[launch defaults] LocalVelocity cavity {res}", flush=True)
    case = cases.cavity3d_local_velocity(res, dtype=np.float32)
    lats = []
    for _ in range(2):
        lat = Lattice(case.extent, case.padding, case.periodic, "f32")
        case.apply(lat)
        lats.append(lat)
    lats[1].set_launch(256, 0)

    def steps(lat):
        for _ in range(20):
            lat.collide_and_stream(1)
        lat.synchronize()

    for lat in lats:
        steps(lat)
    default, uncapped = least([lambda: steps(lats[0]), lambda: steps(lats[1])])
    for lat in lats:
        lat.close()
    assert default <= (1.07 if res == 150 else 1.05) * uncapped
