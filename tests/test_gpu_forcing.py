"""The bound tank's forcing against the oracle where its scheduling changes form:
blade classes merged into one level per radial class or not (by the distance of
the blades at the inner radius, and not where a blade stencil may wrap), levels
on a part of a workgroup, planes whose force values and moments stay in LDS or
not, and the same in batches, whose workgroups have less LDS.  The point order of
the lists fixes every rounding, so results are bit-identical."""
import numpy as np
import pytest

import tdlbcpp_amd as td
from oracle import oracle as O
from tests.helpers import ReferenceLoop, flow_for_tank
from tests.test_gpu_parity import LAYOUTS, STREAMS, random_points, seeded_pair

pytestmark = pytest.mark.gpu


def compare(T, steps, precision, rp=None, streaming=(td.STREAM_ESOTWIST, O.ESOTWIST), angle=0.0):
    dtype = O.F64 if precision == td.PREC_F64 else O.F32
    oflow, gflow = flow_for_tank(T, dtype=dtype)
    o = O.OracleCU(T, dtype=dtype, layout=O.LIJK, streaming=streaming[1], use_les=True, **oflow)
    g = td.ComputeUnit(T, layout=td.LAYOUT_LIJK, streaming=streaming[0], precision=precision, **gflow)
    o.initialise(1.0)
    g.initialise(1.0)
    rp = rp or td.rushton_defaults(T, startup_steps=2)
    g.bind_rushton(rp, angle=angle)
    ref = ReferenceLoop(o, rp, angle=angle, precision=dtype)
    g.run(steps)
    ref.run(steps)
    g.synchronize()
    assert np.array_equal(g.get(td.FIELD_F), o.get(O.FIELD_F)), "F"
    assert np.array_equal(g.get(td.FIELD_Q), o.get(O.FIELD_Q)), "Q"
    g.close()


# 24: a class per blade; 36..50: two colours; from 51 the blades are apart (inner radius T/12)
@pytest.mark.parametrize("T", [12, 24, 36, 50, 51, 52, 97])
@pytest.mark.parametrize("precision", [td.PREC_F32, td.PREC_F64], ids=["fp32", "fp64"])
def test_blade_levels_match_oracle(T, precision):
    print(f"[gpu case] blade levels T={T} precision {precision}", flush=True)
    compare(T, 3, precision, angle=0.3)


def test_simple_streaming_matches_oracle():
    print("[gpu case] forcing, Simple T=53", flush=True)
    compare(53, 3, td.PREC_F32, streaming=(td.STREAM_SIMPLE, O.SIMPLE))


def test_blades_reaching_the_walls_are_not_merged():
    """Blades whose stencils wrap to the other side of the grid meet the opposite blade there."""
    T = 47
    rp = td.rushton_defaults(T, startup_steps=2)
    rp.blade_outer_radius, rp.blade_inner_radius = 23.0, 12.0
    print(f"[gpu case] blades to the walls T={T}", flush=True)
    compare(T, 4, td.PREC_F32, rp=rp)


def wide_disk(T, radius):
    rp = td.rushton_defaults(T, startup_steps=2)
    rp.disk_radius = radius
    return rp


# static cells of the disk plane: about 8500 (force values in LDS, moments not), 16500 (neither)
@pytest.mark.parametrize("T,radius", [(110, 50.0), (150, 70.0)])
def test_planes_beyond_the_lds_match_oracle(T, radius):
    print(f"[gpu case] disk of radius {radius} in {T}^3", flush=True)
    compare(T, 2, td.PREC_F32, rp=wide_disk(T, radius))


def test_fp64_plane_beyond_the_lds_matches_oracle():
    print("[gpu case] disk of radius 50 in 110^3, fp64", flush=True)
    compare(110, 2, td.PREC_F64, rp=wide_disk(110, 50.0))


# workgroups of 64 lanes leave a plane 10 KB of LDS: no room for the blades' rows of the 97^3 tank
@pytest.mark.parametrize("block", [None, "64", "1024"])
def test_batch_levels_match_solo_runs(block, monkeypatch):
    if block:
        monkeypatch.setenv("TDLB_BATCH_FORCE_BLOCK", block)
    print(f"[gpu case] batch levels, block {block}", flush=True)
    specs = [(24, None), (51, None), (97, None), (110, 50.0), (150, 70.0)]

    def tank(T, radius):
        cu = td.ComputeUnit(T, precision=td.PREC_F16, **td.flow_for_tank(T))
        cu.initialise(1.0)
        cu.bind_rushton(wide_disk(T, radius) if radius else td.rushton_defaults(T, startup_steps=2))
        return cu

    batch = td.Batch(td.PREC_F16)
    members = [tank(*s) for s in specs]
    for cu in members:
        batch.add(cu, 5)
    batch.run(5)
    for cu, s in zip(members, specs):
        solo = tank(*s)
        solo.run(5)
        assert np.array_equal(cu.get(td.FIELD_F), solo.get(td.FIELD_F)), s
        assert np.array_equal(cu.get(td.FIELD_Q), solo.get(td.FIELD_Q)), s
        solo.close()
    batch.close()
    for cu in members:
        cu.close()


# A caller's list: more points in a plane than a workgroup has lanes, one cell many times, stencils that meet
# themselves, planes whose cells the LDS has no room for.
@pytest.mark.parametrize("shape,n,same", [((8, 5, 7), 3000, 0), ((6, 3, 70), 600, 700), ((2, 3, 2), 60, 0),
                                          ((200, 2, 200), 3000, 100)])
@pytest.mark.parametrize("precision", [td.PREC_F32, td.PREC_F64], ids=["fp32", "fp64"])
@pytest.mark.parametrize("stream", STREAMS, ids=["Simple", "Esotwist"])
def test_forcing_of_a_list_matches_oracle(shape, n, same, precision, stream):
    print(f"[gpu case] list of {n} + {same} points in {shape}, precision {precision}", flush=True)
    for even in (True, False):
        o, g = seeded_pair(LAYOUTS[0], stream, precision, False, shape=shape, seed=5, even=even)
        rng = np.random.default_rng(6)
        pts = random_points(rng, shape, n + same)
        for axis in "ijk":
            pts[axis][n // 2:n // 2 + same] = pts[axis][0]
        for part in (pts, pts[::3].copy()):
            o.forcing(part, 0.97, 1.9)
            g.forcing(part, 0.97, 1.9)
            np.testing.assert_array_equal(g.get(td.FIELD_F), o.get(O.FIELD_F))
        g.close()
