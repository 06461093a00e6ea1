"""The levels that a tank's blades take, as the library counts them (CPU)."""
import math

import pytest

import tdlbcpp_amd as td
from tests.host_library import host_library  # noqa: F401

# Blades run together, a level per radial class, where neighbouring ones are 3 sqrt(2) cells apart at the inner
# radius: of the default tank from 54 on, but for 58 and 59.  Smaller ones have two colours, the smallest six.
MERGED = {53: False, 54: True, 57: True, 58: False, 59: False, 60: True, 61: True, 97: True}


def expected(T):
    p = td.rushton_defaults(T)
    radial = min(int(math.floor(p.blade_outer_radius - p.blade_inner_radius + 1e-9)) + 1, 5)
    apart = 2 * p.blade_inner_radius * math.sin(math.pi / 6) >= 3 * math.sqrt(2) + 1e-9
    two = 2 * p.blade_inner_radius * math.sin(math.pi * 2 / 6) >= 3 * math.sqrt(2) + 1e-9
    return radial * (1 if apart else 2 if two else 6), apart


@pytest.mark.parametrize("T", sorted(MERGED))
def test_blades_merge_by_their_distance(T):
    assert expected(T)[1] == MERGED[T]


def test_forcing_info_counts_the_levels_that_run(host_library):  # noqa: F811
    """One static level (the host library's kernels find no other) and the blade levels."""
    sizes = [12, 24, 30, 36, 50, 53, 54, 57, 58, 59, 60, 97, 128]
    want = {T: expected(T)[0] for T in sizes}
    assert want[24] == 18 and want[60] == 5 and want[97] == 5 and want[53] == 10
    host_library(f"""
    for T, blades in {want!r}.items():
        cu = tank(T)
        assert cu.forcing_info()[2] == 1 + blades, (T, cu.forcing_info(), blades)
        cu.close()
    # blades whose stencils wrap are never merged
    rp = td.rushton_defaults(60)
    rp.blade_outer_radius, rp.blade_inner_radius = 29.0, 20.0
    cu = tank(60, bind=False)
    cu.bind_rushton(rp)
    assert cu.forcing_info()[2] == 1 + 10
    cu.close()
    """)
