"""Moments of lattices on threads and streams of their own: a call waits for the
work of its own stream only, not for another thread's, and concurrent calls, on
one lattice too, return what calls one after another do."""
import threading
import time
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from openlb_amd import Lattice, cases

pytestmark = pytest.mark.gpu


def _lattice(n):
    case = cases.tgv(n, dtype=np.float32)
    lat = Lattice(case.extent, case.padding, case.periodic, "f32")
    case.apply(lat)
    return lat


def test_moments_do_not_wait_for_another_lattice():
    print("[moments] two threads", flush=True)
    busy, idle = _lattice(256), _lattice(40)
    own = [torch.cuda.Stream(), torch.cuda.Stream()]
    busy.set_two_step(0)
    for lat, stream in zip((busy, idle), own):
        lat.collide_and_stream(2, stream.cuda_stream)
        lat.reduce_moments(stream.cuda_stream)
    took = []

    def work():
        t = time.perf_counter()
        busy.collide_and_stream(400, own[0].cuda_stream)
        busy.reduce_moments(own[0].cuda_stream)
        took.append(time.perf_counter() - t)

    thread = threading.Thread(target=work)
    thread.start()
    time.sleep(0.03)
    t = time.perf_counter()
    got = idle.reduce_moments(own[1].cuda_stream)
    waited = time.perf_counter() - t
    thread.join()
    assert got == idle.reduce_moments(own[1].cuda_stream)
    busy.close()
    idle.close()
    # 400 steps take 200 ms; the other call shares the chip with two or three of them
    assert took[0] > 0.12 and waited < 0.25 * took[0]


def test_concurrent_moments_agree():
    print("[moments] eight threads", flush=True)
    lats = [_lattice(n) for n in (16, 40, 64, 101)]
    for lat in lats:
        lat.collide_and_stream(3)
        lat.synchronize()
    want = [lat.reduce_moments() for lat in lats]
    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(lambda k: lats[k % 4].reduce_moments(), range(64)))
    assert got == [want[k % 4] for k in range(64)]
    for lat in lats:
        lat.close()
