"""The vorticity pictures against the oracle up to the edges of the grid, where the
central differences read ghost cells (the far-side ones of Esotwist are undefined in
the reference and NaN here)."""
import numpy as np
import pytest

import tdlbcpp_amd as td
from oracle import oracle as O
from tests.test_gpu_parity import STREAMS, seeded_pair

pytestmark = pytest.mark.gpu

LAYOUTS = [(td.LAYOUT_IJKL, O.IJKL), (td.LAYOUT_LIJK, O.LIJK), (td.LAYOUT_IJKL_SOA, O.IJKL)]


# the logarithms of the device and the host differ in the last places
@pytest.mark.parametrize("precision,rtol", [(td.PREC_F32, 2e-6), (td.PREC_F64, 1e-14)], ids=["fp32", "fp64"])
@pytest.mark.parametrize("layout", LAYOUTS, ids=["IJKL", "LIJK", "IJKL_SOA"])
@pytest.mark.parametrize("stream", STREAMS, ids=["Simple", "Esotwist"])
def test_vorticity_at_the_edges_matches_oracle(stream, layout, precision, rtol):
    for shape in ((7, 6, 9), (66, 3, 70)):
        for even in (True, False):
            print(f"[gpu case] vorticity {shape} {stream} {layout} precision {precision} even {even}", flush=True)
            o, g = seeded_pair(layout, stream, precision, True, shape=shape, seed=4, even=even)
            for axis, last in ((0, shape[1]), (1, shape[2])):
                for cut in sorted({1, 2, last // 2 + 1, last}):
                    gv, ov = g.vorticity(axis, cut), o.vorticity(axis, cut)
                    np.testing.assert_array_equal(np.isnan(gv), np.isnan(ov))
                    some = ~np.isnan(ov)
                    np.testing.assert_allclose(gv[some], ov[some], rtol=rtol)
            g.close()
