"""The bound tank's forcing against the oracle at both sides of the rules that choose
its form: blades merged into one level per radial class or not, a plane in two tasks,
levels found at bind with a plane's marks in HBM."""
import numpy as np
import pytest

import tdlbcpp_amd as td
from tests.test_forcing_levels import MERGED
from tests.test_gpu_forcing import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", sorted(MERGED))
def test_blades_around_the_merging_rule_match_oracle(T):
    print(f"[gpu case] blades {'merged' if MERGED[T] else 'by colour'} T={T} fp32", flush=True)
    compare(T, 3, td.PREC_F32, angle=0.3)


@pytest.mark.parametrize("T", [54, 58])
def test_blades_around_the_merging_rule_match_oracle_fp64(T):
    print(f"[gpu case] blades {'merged' if MERGED[T] else 'by colour'} T={T} fp64", flush=True)
    compare(T, 3, td.PREC_F64, angle=0.3)


def disk_plane_cells(T):
    """Unique static stencil cells of the impeller disk's plane."""
    p = td.rushton_defaults(T)
    pts = np.concatenate([td.rushton_generate(p, td.GEOM_FIXED),
                          td.rushton_generate(p, td.GEOM_ROTATING_NON_UPDATING, 0.0, 0.01)])
    pts = pts[pts["j"] == p.disk_plane]
    i = (pts["i"][:, None] + np.array([-1, 0, 1] * 3)) % T
    k = (pts["k"][:, None] + np.repeat([-1, 0, 1], 3)) % T
    return len(np.unique(i * T + k))


def test_plane_in_two_tasks_matches_oracle_fp64():
    """The disk and the wall of a plane share no cell and together exceed the LDS (160 KB, 7 doubles a cell)."""
    T = 160
    assert disk_plane_cells(T) * 7 * 8 > 160 * 1024
    print(f"[gpu case] disk plane in two tasks T={T} fp64", flush=True)
    compare(T, 2, td.PREC_F64)


def test_levels_with_marks_in_hbm_match_oracle():
    """200^2 marks exceed the 152 KB of LDS that the level search at bind may take."""
    T = 200
    assert T * T * 4 > 152 * 1024
    print(f"[gpu case] levels at bind with marks in HBM T={T} fp32", flush=True)
    compare(T, 1, td.PREC_F32)
