"""The bound tank's forcing against the oracle where its scheduling changes form:
blade classes merged into one level per radial class or not (by the distance of
the blades at the inner radius, and not where a blade stencil may wrap), levels
on a part of a workgroup, planes whose force values stay in LDS or not.  The
point order of the lists fixes every rounding, so results are bit-identical."""
import numpy as np
import pytest

import tdlbcpp_amd as td
from oracle import oracle as O
from tests.helpers import ReferenceLoop, flow_for_tank

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
