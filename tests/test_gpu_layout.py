"""Q at the boundary: every value of a lattice larger than one staging piece comes
back from HBM where it was put, ghosts included, in both orders, and one cell is
the same cell in both."""
import numpy as np
import pytest

import tdlbcpp_amd as td

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 7, 66), (33, 190, 1003)])
@pytest.mark.parametrize("precision", [td.PREC_F32, td.PREC_F64], ids=["fp32", "fp64"])
def test_q_round_trip(dims, precision):
    print(f"[gpu case] Q round trip {dims} precision {precision}", flush=True)
    word = np.uint64 if precision == td.PREC_F64 else np.uint32
    values = None
    for layout in (td.LAYOUT_IJKL, td.LAYOUT_LIJK, td.LAYOUT_IJKL_SOA):
        cu = td.ComputeUnit(*dims, layout=layout, streaming=td.STREAM_ESOTWIST, precision=precision)
        n = cu.field_bytes(td.FIELD_Q) // np.dtype(cu.np_dtype).itemsize
        if values is None:
            values = np.arange(n, dtype=word).reshape(cu.xg, cu.yg, cu.zg, 18)
        cu.set_q_ijkl(values.view(cu.np_dtype))
        assert np.array_equal(cu.q_ijkl().view(word) if layout != td.LAYOUT_LIJK
                              else np.ascontiguousarray(cu.q_ijkl()).view(word), values), layout
        cu.close()
