"""Addresses past 2^32: a tank at the far end of a grid whose last slot plane lies past
2^32 elements advances as the same tank in a small grid, and the rest of the grid stays
at rest.  (Esotwist is periodic and a step reaches one cell further, so a few steps do
not reach the edges of either grid.)"""
import numpy as np
import pytest

import tdlbcpp_amd as td

pytestmark = pytest.mark.gpu

T, STEPS = 36, 4
SMALL, BIG = (64, 64, 64), (1000, 490, 490)
FAR = (940, 440)  # lower corner of the tank in the big grid, in i and k
AT = (13, 14)     # and in the small one: the order of the lists goes by the points' i mod 3 and k mod 3
assert all((f - a) % 3 == 0 for f, a in zip(FAR, AT))


ANGLE = 0.1       # blades at 0 have points halfway between cells, which fall to either side by rounding


def geometry(corner):
    rp = td.rushton_defaults(T, tip_speed=0.1, startup_steps=0)
    rp.center_x += corner[0]
    rp.center_z += corner[1]
    return rp


def lists(corner):
    """Every point list of the run: the static ones, and the blades at bind and after each step"""
    rp, d = geometry(corner), float(np.float32(td.rushton_step_increment(geometry(corner), 1)))
    return [td.rushton_generate(rp, td.GEOM_FIXED), td.rushton_generate(rp, td.GEOM_ROTATING_NON_UPDATING, 0.0, d)] + \
           [td.rushton_generate(rp, td.GEOM_ROTATING, ANGLE + n * d, d) for n in range(STEPS + 1)]


def field(shape, corner, layout, precision):
    flow = td.flow_for_tank(T, re=1.0e4, uav=0.1, cs0=0.1, use_les=1)
    cu = td.ComputeUnit(*shape, layout=layout, precision=precision, **flow)
    cu.initialise(1.0)
    cu.bind_rushton(geometry(corner), angle=ANGLE)
    cu.run(STEPS)
    out = cu.macroscopic()
    cu.close()
    return out


# Positions differ by the rounding of i + 927 in doubles, fractions so by at most an ulp of a float (6e-8), weights
# (slope at most 1, sums of nine) and forces (0.1 at most) by a few times that a step: 2e-6 is ten times as much.  A
# 16-bit population may round the other way: half an ulp of fp16 of a deviation of 0.05 each, 2e-5, nine of them.
@pytest.mark.parametrize("layout,precision,tol", [(td.LAYOUT_LIJK, td.PREC_F32, 2e-6), (td.LAYOUT_IJKL, td.PREC_F32, 2e-6),
                                                  (td.LAYOUT_LIJK, td.PREC_F16, 2e-4)])
def test_tank_past_2_32_elements_equals_the_tank_in_a_small_grid(layout, precision, tol):
    print(f"[gpu case] tank of {T} at {FAR} in {BIG}, layout {layout} precision {precision}", flush=True)
    cells = np.prod([n + 2 for n in BIG])
    assert 17 * cells + FAR[0] * (BIG[1] + 2) * BIG[2] > 2 ** 32
    for a, b in zip(lists(AT), lists(FAR)):  # the same tank: every point in the same cell of it, in the same order
        assert (b["i"] - a["i"] == FAR[0] - AT[0]).all() and (b["k"] - a["k"] == FAR[1] - AT[1]).all()
    small = field(SMALL, AT, layout, precision)
    big = field(BIG, FAR, layout, precision)
    assert np.abs(small[..., 1:]).max() > 0.02
    di, dk = FAR[0] - AT[0], FAR[1] - AT[1]
    reach = STEPS + 2
    tank = big[di:di + SMALL[0], :, dk:dk + SMALL[2]]
    up = T + reach
    np.testing.assert_allclose(tank[:, :up], small[:, :up], rtol=0, atol=tol)
    np.testing.assert_allclose(tank[:, BIG[1] - reach:], small[:, SMALL[1] - reach:], rtol=0, atol=tol)
    # everything further away than the steps reach: the rest state of the small grid's far corner
    rest = small[0, SMALL[1] - reach - 8, 0]
    near = (slice(FAR[0] - reach, FAR[0] + T + reach), slice(FAR[1] - reach, FAR[1] + T + reach))
    big[near[0], :up, near[1]] = rest
    big[near[0], BIG[1] - reach:, near[1]] = rest
    for i in range(0, BIG[0], 50):
        assert (big[i:i + 50] == rest).all(), i
