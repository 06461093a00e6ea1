"""Q at the boundary: every value of a lattice larger than one staging piece comes
back from HBM where it was put, ghosts included, in both orders, and one cell is
the same cell in both."""
import numpy as np
import pytest

import tdlbcpp_amd as td
from oracle import oracle as O
from tests.test_gpu_forcing import compare

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


def test_results_read_by_several_threads_at_once():
    """Six threads, each with a handle and stream of its own, share the pinned buffers of the read-back
    (four of each size): every field equals the one read alone."""
    import threading
    edges = (24, 37, 64, 65, 90, 101)
    cus = []
    for n, e in enumerate(edges):
        cu = td.ComputeUnit(e, precision=td.PREC_F16 if n % 2 else td.PREC_F32, **td.flow_for_tank(e))
        cu.initialise(1.0)
        cu.bind_rushton(td.rushton_defaults(e, startup_steps=2))
        cu.run(3)
        cus.append(cu)
    for cu in cus:
        cu.get(td.FIELD_F)  # leaves the handle with its moments stored, as every later read finds it
    alone = [(cu.macroscopic(), cu.get(td.FIELD_F), cu.get(td.FIELD_NU)) for cu in cus]
    got = [None] * len(cus)
    print("[gpu case] read-back from six threads", flush=True)

    def read(n):
        got[n] = [(cus[n].macroscopic(), cus[n].get(td.FIELD_F), cus[n].get(td.FIELD_NU)) for _ in range(3)]

    threads = [threading.Thread(target=read, args=(n,)) for n in range(len(cus))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        assert b is not None
        for r in b:
            assert all(np.array_equal(x, y) for x, y in zip(a, r))
    for cu in cus:
        cu.close()


# Rows that end inside a wavefront: the fused step takes the cells of a plane back to back (a row of one
# cell more than a wavefront, of an odd size, and FP64 rows within one wavefront, which stay rows).
@pytest.mark.parametrize("T", [30, 65, 71, 116])
@pytest.mark.parametrize("precision", [td.PREC_F32, td.PREC_F64], ids=["fp32", "fp64"])
@pytest.mark.parametrize("streaming", [(td.STREAM_ESOTWIST, O.ESOTWIST), (td.STREAM_SIMPLE, O.SIMPLE)],
                         ids=["Esotwist", "Simple"])
def test_rows_ending_inside_a_wavefront_match_oracle(T, precision, streaming):
    print(f"[gpu case] rows of {T}, precision {precision}", flush=True)
    compare(T, 3, precision, streaming=streaming)


# one launch writes every face and edge: rims where faces meet, extents of one cell
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 4, 2), (3, 1, 5), (66, 3, 2), (5, 6, 130)])
@pytest.mark.parametrize("precision", [td.PREC_F32, td.PREC_F64], ids=["fp32", "fp64"])
def test_bounce_back_of_all_faces_matches_oracle(shape, precision):
    print(f"[gpu case] bounce-back {shape}, precision {precision}", flush=True)
    o = O.OracleCU(*shape, dtype=O.F32 if precision == td.PREC_F32 else O.F64, layout=O.LIJK, streaming=O.SIMPLE,
                   use_les=False, nu=0.003)
    g = td.ComputeUnit(*shape, layout=td.LAYOUT_LIJK, streaming=td.STREAM_SIMPLE, precision=precision, nu=0.003)
    q = np.random.default_rng(3).standard_normal(o.get(O.FIELD_Q).shape)
    o.set(O.FIELD_Q, q)
    g.set(td.FIELD_Q, o.get(O.FIELD_Q))
    for _ in range(2):
        o.bounce_back()
        g.bounce_back()
        assert np.array_equal(g.get(td.FIELD_Q), o.get(O.FIELD_Q))
        o.streaming_push()
        g.streaming_push()
    g.close()
