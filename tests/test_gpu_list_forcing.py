"""The forcing of a caller's list from several threads, and in grids of many planes."""
import threading

import numpy as np
import pytest

import tdlbcpp_amd as td
from tests.test_gpu_parity import random_points

pytestmark = pytest.mark.gpu


def forced(shape, n, seed, calls):
    """F after `calls` forcing calls of random lists on a fresh handle"""
    rng = np.random.default_rng(seed)
    cu = td.ComputeUnit(*shape)
    cu.initialise(1.0)
    for _ in range(calls):
        cu.forcing(random_points(rng, shape, n), 0.97, 1.9)
    out = cu.get(td.FIELD_F)
    cu.close()
    return out


def test_threads_with_planes_of_different_sizes():
    """Planes whose marks take 68, 110 and 150 KB of LDS, forced from a thread each at the same time: every launch
    has the LDS it asks for, and the results are those of the same calls one after the other."""
    shapes = [(130, 2, 130), (166, 2, 166), (194, 2, 194)]
    print(f"[gpu case] lists from {len(shapes)} threads, {shapes}", flush=True)
    want = [forced(s, 400, n, 12) for n, s in enumerate(shapes)]
    got = [None] * len(shapes)
    start = threading.Barrier(len(shapes))

    def work(n):
        start.wait()
        got[n] = forced(shapes[n], 400, n, 12)

    threads = [threading.Thread(target=work, args=(n,)) for n in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for w, g in zip(want, got):
        np.testing.assert_array_equal(g, w)
