"""The forcing of a caller's list from several threads, and in grids of many planes."""
import threading

import numpy as np
import pytest

import tdlbcpp_amd as td
from oracle import oracle as O
from tests.test_gpu_parity import LAYOUTS, STREAMS, random_points, seeded_pair

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


# more planes than workgroups, most of them without points: a few in every so many planes, in the last ones only,
# in all
@pytest.mark.parametrize("n,planes", [(300, None), (40, (8990, 9000)), (1, (0, 1)), (30000, None)])
def test_many_planes_match_oracle(n, planes):
    shape = (5, 9000, 6)
    print(f"[gpu case] list of {n} points in {shape}, planes {planes}", flush=True)
    o, g = seeded_pair(LAYOUTS[0], STREAMS[1], td.PREC_F32, False, shape=shape, seed=3, even=True)
    rng = np.random.default_rng(n)
    for _ in range(2):
        pts = random_points(rng, shape, n)
        if planes:
            pts["j"] = rng.integers(planes[0], planes[1], n)
        o.forcing(pts, 0.97, 1.9)
        g.forcing(pts, 0.97, 1.9)
        np.testing.assert_array_equal(g.get(td.FIELD_F), o.get(O.FIELD_F))
    g.close()
