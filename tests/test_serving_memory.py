"""The server's account of device memory (CPU, tests/host)."""
import pytest

from tests.host_library import host_library  # noqa: F401

DRAIN = """
def drain(s):
    done, most = [], 0
    for _ in range(100000):
        resident, queued, _ = s.tick()
        most = max(most, resident)
        done += s.poll()
        if resident == 0 and queued == 0:
            return done, most
    raise SystemExit("server did not drain")
"""


@pytest.mark.parametrize("prec", ["F16", "F32", "E3M12"])
@pytest.mark.parametrize("stream", ["ESOTWIST", "SIMPLE"])
def test_a_tank_holds_no_more_than_is_reserved_for_it(host_library, prec, stream):  # noqa: F811
    """The most that a tank holds from its first allocation to its result is at most what admission reserves."""
    host_library(DRAIN, f"""
    for edge in (12, 17, 24, 30, 48, 64, 81, 96, 128, 160, 197):
        s = td.Server(td.PREC_{prec}, td.LAYOUT_LIJK, td.STREAM_{stream}, tick_steps=50)
        L.fake_reset_peak()
        start = L.fake_live()
        s.submit(edge, 0.1, 5000.0, 120)
        s.tick()
        reserved = s.stats()["reserved_bytes"]
        done, _ = drain(s)
        assert done[0]["error"] == 0
        assert L.fake_peak() - start <= reserved, (edge, L.fake_peak() - start, reserved)
        s.close()
        assert L.fake_live() == 0
    """)


def test_admission_counts_every_tank(host_library):  # noqa: F811
    """Tanks of 64^3 run together only as far as the budget holds what they take, and every request that fitted
    the budget by its lattice is served, alone if need be."""
    host_library(DRAIN, """
    def lattice(edge):  # what a request may not exceed the budget by: lattices, F, Nu, O, masks, and 10 %
        lo, hi = 1, 1 << 32
        while lo < hi:
            mid = (lo + hi) // 2
            t = td.Server(td.PREC_F16, hbm_budget=float(mid))
            try:
                t.submit(edge, 0.1, 5000.0, 3)
                hi = mid
            except td.TdlbError:
                lo = mid + 1
            t.close()
        return lo
    one = lattice(64)
    n = 66 ** 3
    assert one >= 1.1 * n * (36 + 12 + 2 + 1) * 0.9
    for budget in (one, 3.05 * one):
        s = td.Server(td.PREC_F16, hbm_budget=float(budget), tick_steps=10)
        L.fake_reset_peak()
        start = L.fake_live()
        for _ in range(4):
            s.submit(64, 0.1, 5000.0, 30000)
        done, most = drain(s)
        assert len(done) == 4 and all(r["error"] == 0 for r in done)
        if budget > one:
            assert most >= 2 and L.fake_peak() - start <= budget, (most, L.fake_peak() - start, budget)
        assert s.stats()["reserved_bytes"] == 0
        s.close()
    """)
