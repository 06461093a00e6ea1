"""A bind that fails leaves no half-made geometry to run on (CPU)."""
from tests.host_library import host_library  # noqa: F401


def test_failed_rebind_leaves_the_handle_unbound(host_library):  # noqa: F811
    """Whichever allocation of a second bind fails: run and batches refuse the handle (TDLB_ERR_STATE), no
    forcing is launched on it, and a bind that succeeds makes it runnable again."""
    host_library("""
    rp = td.rushton_defaults(36)
    one, ang = ctypes.c_uint64(1), ctypes.c_double(0.0)
    n = 0
    while True:
        cu = td.ComputeUnit(48)
        cu.initialise(1.0)
        cu.bind_rushton(td.rushton_defaults(24))  # fewer points than the second geometry: its buffers grow
        batch, other = td.Batch(td.PREC_F32), td.Batch(td.PREC_F32)
        batch.add(cu, 1000)
        batch.run(2)
        L.fake_fail_malloc(n)
        rc = L.tdlb_cu_bind_rushton(cu._h, ctypes.byref(rp), 1, 0.0, 0.97, 1.9)
        L.fake_fail_malloc(-1)
        if rc != 0:
            assert rc == NOMEM, rc
            before = L.fake_gathers()
            assert L.tdlb_cu_run(cu._h, 1, ctypes.byref(one), ctypes.byref(ang)) == STATE, n
            assert L.tdlb_batch_run(batch._b, 1, None) == STATE, n
            assert L.tdlb_batch_add(other._b, cu._h, 1, 0.0, 5) == STATE, n
            assert L.fake_gathers() == before
            cu.bind_rushton(rp)
        cu.run(1)
        batch.run(1)
        batch.close()
        other.close()
        cu.close()
        if rc == 0:
            break
        n += 1
    assert n > 8
    """)


def test_refused_rebind_keeps_the_earlier_geometry(host_library):  # noqa: F811
    """Arguments that are refused are refused before anything of the bound geometry changes."""
    host_library("""
    cu = tank(36)
    info = cu.forcing_info()
    rp = td.rushton_defaults(36)
    rp.n_blades = 17
    try:
        cu.bind_rushton(rp)
        raise SystemExit("17 blades accepted")
    except td.TdlbError:
        pass
    cu.run(2)
    assert cu.forcing_info() == info
    cu.close()
    """)


def test_marks_of_large_planes_take_what_memory_there_is(host_library):  # noqa: F811
    """A plane beyond the LDS has its marks in HBM, a plane a workgroup: with little memory left a bind and a
    forcing call run with fewer workgroups, and with no room for one plane they are TDLB_ERR_NOMEM."""
    host_library("""
    def grid():
        cu = td.ComputeUnit(220, 60, 220)
        cu.initialise(1.0)
        return cu
    plane = 220 * 220 * 4
    rp = td.rushton_defaults(60)
    cu = grid()
    L.fake_reset_peak()
    start = L.fake_live()
    cu.bind_rushton(rp)
    tank_bytes = L.fake_live() - start        # what stays
    assert L.fake_peak() - start > 60 * plane
    n_static = cu.forcing_info()[0]
    pts = td.rushton_generate(rp, td.GEOM_FIXED)
    cu.forcing(pts, 0.97, 1.9)
    assert L.fake_live() - start > tank_bytes + 60 * plane
    cu.close()
    assert tank_bytes < 45 * plane
    for room, ok in ((20 * plane, True), (plane + 100, True), (plane - 1000, False)):
        cu = grid()
        # what stays and the transients of its tables; or the list's positions, indices and levels
        few = n_static * 24 + room
        L.fake_limit(L.fake_live() + (max(few, tank_bytes + n_static * 36 + cu.xg * cu.yg * 32) if ok else few))
        rc = L.tdlb_cu_bind_rushton(cu._h, ctypes.byref(rp), 1, 0.0, 0.97, 1.9)
        L.fake_limit(1 << 40)
        assert rc == (0 if ok else NOMEM), (room, rc)
        cu.close()
        cu = grid()
        L.fake_limit(L.fake_live() + len(pts) * (64 + 8 + 12 + 20) + room)
        p = np.ascontiguousarray(pts)
        for _ in range(2):
            rc = L.tdlb_cu_forcing(cu._h, p.ctypes.data, len(p), 0.97, 1.9)
            assert rc == (0 if ok else NOMEM), (room, rc)
        L.fake_limit(1 << 40)
        cu.forcing(pts, 0.97, 1.9)
        cu.close()
        assert L.fake_live() == 0
    """)


def test_a_call_after_an_allocation_that_failed(host_library):  # noqa: F811
    """TDLB_ERR_NOMEM is the error of its own call: the next call on the thread, with memory again, succeeds."""
    host_library("""
    pts = np.ascontiguousarray(td.rushton_generate(td.rushton_defaults(24), td.GEOM_FIXED))
    rp = td.rushton_defaults(24)
    out = (ctypes.c_double * 8)()
    for n in range(3):
        cu, half = tank(24, bind=False), tank(24, td.PREC_F16, bind=False)
        batch = td.Batch(td.PREC_F32)
        nu = np.zeros(half.size, dtype=np.float32)
        solid = np.zeros(cu.size, dtype=np.uint8)
        bound = tank(24)
        def calls():
            yield L.tdlb_cu_forcing(cu._h, pts.ctypes.data, len(pts), 0.97, 1.9)
            yield L.tdlb_cu_reductions(cu._h, out)
            yield L.tdlb_cu_upload(half._h, td.FIELD_NU, nu.ctypes.data, nu.nbytes)
            yield L.tdlb_cu_solid_mask(bound._h, solid.ctypes.data, solid.nbytes)
            yield L.tdlb_batch_add(batch._b, bound._h, 1, 0.0, 5)
            yield L.tdlb_cu_bind_rushton(cu._h, ctypes.byref(rp), 1, 0.0, 0.97, 1.9)
        it = calls()
        while True:
            L.fake_fail_malloc(n)
            rc = next(it, None)
            L.fake_fail_malloc(-1)
            if rc is None:
                break
            assert rc in (0, NOMEM), rc
            assert L.tdlb_cu_collision(cu._h) == 0, rc
        batch.close()
        for c in (cu, half, bound):
            c.close()
    """)
