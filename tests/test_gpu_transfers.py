"""Uploads and downloads from several threads, whose pieces of device memory and pinned
buffers are shared, with handles that come and go in between."""
import threading

import numpy as np
import pytest

import tdlbcpp_amd as td

pytestmark = pytest.mark.gpu


def test_threads_upload_and_download_at_once():
    """Five threads, a handle each, sizes of one piece and of several: every Q, F and Nu comes back as it was put."""
    cases = [(12, td.LAYOUT_IJKL, td.PREC_F32), (30, td.LAYOUT_IJKL, td.PREC_F64), (61, td.LAYOUT_LIJK, td.PREC_F32),
             (75, td.LAYOUT_IJKL, td.PREC_F64), (20, td.LAYOUT_IJKL_SOA, td.PREC_F32)]
    print("[gpu case] uploads and downloads from five threads", flush=True)
    start, wrong = threading.Barrier(len(cases)), []

    def work(n):
        edge, layout, precision = cases[n]
        start.wait()
        for turn in range(3):
            with td.ComputeUnit(edge, layout=layout, precision=precision) as cu:
                cu.initialise(1.0)
                for field in (td.FIELD_Q, td.FIELD_NU, td.FIELD_F):
                    size = cu.field_bytes(field) // np.dtype(cu.np_dtype).itemsize
                    a = np.arange(1, size + 1).astype(cu.np_dtype) + turn
                    for _ in range(2):
                        cu.set(field, a)
                        if not np.array_equal(cu.get(field), a):
                            wrong.append((n, turn, field))

    threads = [threading.Thread(target=work, args=(n,)) for n in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
