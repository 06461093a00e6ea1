"""Results to the host when memory or threads are short (CPU, tests/host)."""
import pytest

from tests.host_library import host_library  # noqa: F401

CHECK = """
def check(cu):
    a = cu.macroscopic()
    t = np.arange(a.size // 4, dtype=np.float64)
    want = (t[:, None] + 0.25 * np.arange(4)).astype(a.dtype)
    assert np.array_equal(a.reshape(-1, 4), want)
    for f in (td.FIELD_F, td.FIELD_NU, td.FIELD_O, td.FIELD_Q):
        v = np.random.default_rng(f).integers(0, 200, cu.field_bytes(f) // np.dtype(
            np.uint8 if f == td.FIELD_O else cu.np_dtype).itemsize).astype(np.uint8 if f == td.FIELD_O else cu.np_dtype)
        cu.set(f, v)
        assert np.array_equal(cu.get(f), v), f
"""


# small results and large ones, of a piece and of many; FP64 cells divide no power of two evenly
@pytest.mark.parametrize("T,prec", [(6, "F32"), (17, "F64"), (70, "F32"), (101, "F64")])
@pytest.mark.parametrize("pinned", [-1, -2, 1])
def test_results_come_without_pinned_memory(host_library, T, prec, pinned):  # noqa: F811
    """Every result comes back whole when pinned memory is there (-1), never there (-2) or gone after the first
    buffer (1), and the failed allocation is no error of a later call."""
    host_library(CHECK, f"""
    L.fake_fail_pinned({pinned})
    cu = tank({T}, td.PREC_{prec}, bind=False)
    for _ in range(3):
        check(cu)
        cu.collision()
    cu.close()
    assert L.fake_live() == 0 and L.fake_pinned() == 0
    """)


def test_results_come_in_small_pieces_of_device_memory(host_library):  # noqa: F811
    """Without pinned memory and with little device memory the pieces get smaller; with none TDLB_ERR_NOMEM."""
    host_library("""
    L.fake_fail_pinned(-2)
    out = np.empty((128, 128, 128, 4), dtype=np.float32)
    for room, rc in ((1 << 40, 0), (3 << 20, 0), (1 << 10, NOMEM)):
        L.fake_limit(1 << 40)
        cu = tank(128, bind=False)
        L.fake_limit(L.fake_live() + room)
        out[:] = -1
        assert L.tdlb_cu_macroscopic(cu._h, out.ctypes.data, out.nbytes) == rc
        if rc == 0:
            t = np.arange(128 ** 3, dtype=np.float32)
            assert np.array_equal(out.reshape(-1, 4)[:, 0], t)
        o = np.empty(130 ** 3, dtype=np.uint8)  # an array that lies in device memory as it is needs none
        assert L.tdlb_cu_download(cu._h, td.FIELD_O, o.ctypes.data, o.nbytes) == 0
        cu.close()
    assert L.fake_live() == 0
    """)


@pytest.mark.parametrize("n", range(0, 12))
def test_host_memory_short_while_threads_start(host_library, n):  # noqa: F811
    """The n-th host allocation of a read fails: the result comes all the same, and no exception leaves a C call."""
    host_library(CHECK, f"""
    cu = tank(101, td.PREC_F64, bind=False)
    out = np.empty((101, 101, 101, 4))
    for _ in range(4):
        out[:] = -1
        L.fake_fail_new({n})
        rc = L.tdlb_cu_macroscopic(cu._h, out.ctypes.data, out.nbytes)
        L.fake_fail_new(-1)
        assert rc == 0
        assert np.array_equal(out.reshape(-1, 4)[:, 0], np.arange(101 ** 3))
    cu.close()
    """)


def test_pinned_memory_is_made_where_it_pays(host_library):  # noqa: F811
    """Programs that read little between their first handle and their last make no pinned memory; it is given
    back with the last handle, and arrays that lie in device memory as they are do without while small."""
    host_library("""
    def reads(T, n, read, want):
        L.fake_limit(1 << 40)
        before, cu = L.fake_pinned_mallocs(), tank(T, bind=False)
        for _ in range(n):
            read(cu)
        assert L.fake_pinned_mallocs() - before == want, (T, n, L.fake_pinned_mallocs() - before)
        cu.close()
        assert L.fake_pinned() == 0
    field = lambda cu: cu.macroscopic()
    for _ in range(2):
        reads(36, 3, field, 0)
        reads(36, 9, field, 1)
        reads(80, 3, field, 0)     # 8.2 MB each: from 64 MiB on
        reads(80, 9, field, 1)
        reads(96, 1, field, 1)     # 14 MB
        reads(30, 20, lambda cu: cu.get(td.FIELD_O), 0)
        reads(60, 20, lambda cu: cu.get(td.FIELD_O), 0)
        reads(60, 20, lambda cu: cu.get(td.FIELD_NU), 1)
    a, b = tank(36, bind=False), tank(36, bind=False)
    for _ in range(4):
        a.macroscopic()
    a.close()
    assert L.fake_pinned() == 1    # the other handle's reads find it
    b.macroscopic()
    b.close()
    assert L.fake_pinned() == 0 and L.fake_live() == 0
    """)


def test_a_server_keeps_the_buffers_between_its_tanks(host_library):  # noqa: F811
    """Tanks of a server come and go; its reads make the pinned buffers once, and they go with the server."""
    host_library("""
    s = td.Server(td.PREC_F16, tick_steps=50, keep_handles=True)
    for n in range(3):
        t = s.submit(100, 0.1, 5000.0, 20)
        while not s.poll():
            s.tick()
        cu = s.take(t, 100)
        cu.macroscopic()
        cu.close()
        assert L.fake_pinned() == 1 and L.fake_pinned_mallocs() == 1
    s.close()
    assert L.fake_pinned() == 0 and L.fake_live() == 0
    """)


def test_uploads_and_plain_reads_share_a_stage(host_library):  # noqa: F811
    """Uploads of Q and results without pinned memory allocate a piece of device memory the first times and then
    share one, whatever the number of handles and sizes; short memory makes the pieces smaller, none is
    TDLB_ERR_NOMEM, and the piece goes with the last handle."""
    host_library("""
    a, b = tank(30, td.PREC_F64, bind=False), tank(70, bind=False)
    def upload(cu):
        q = np.random.default_rng(1).random(cu.field_bytes(td.FIELD_Q) // np.dtype(cu.np_dtype).itemsize).astype(cu.np_dtype)
        cu.set(td.FIELD_Q, q)
        assert np.array_equal(cu.get(td.FIELD_Q), q)
    n = L.fake_mallocs()
    for _ in range(6):
        upload(a)
        upload(b)
        b.macroscopic()
    assert n < L.fake_mallocs() <= n + 4
    a.close()
    b.close()
    assert L.fake_live() == 0
    b = tank(70, bind=False)
    L.fake_limit(L.fake_live() + (3 << 20))
    upload(b)
    L.fake_limit(L.fake_live() + 1000)
    q = np.zeros(b.field_bytes(td.FIELD_Q) // 4, dtype=np.float32)
    assert L.tdlb_cu_upload(b._h, td.FIELD_Q, q.ctypes.data, q.nbytes) == NOMEM
    b.close()
    assert L.fake_live() == 0
    """)
