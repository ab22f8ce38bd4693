"""The autotuner times what its digit widths are used for: radix passes, also at
the sizes whose unfixed builds merge sorted tiles (batches read those entries, and
larger sizes the nearest one)."""
import pytest

pytestmark = pytest.mark.gpu


def test_widths_are_timed_on_radix_passes(lb):
    reps, buckets = 2, [1 << 11, 1 << 12, 1 << 13]
    with lb.Context(0) as c:
        c.profile_enable()
        times = c.autotune(buckets[0], buckets[-1], reps=reps)
        got = {s: n for s, (_, n) in c.profile_read().items()}
        assert sorted(times) == buckets
        builds = len(buckets) * (reps + 1)  # of each variant, a warm-up too
        # three tiles with each width: 10-bit digits take three passes, 8-bit four
        assert (got["sort2"], got["sort3"]) == (6 * builds, 3 * builds)
        # and unfixed builds of the same sizes merge
        n = buckets[1]
        c.build_arrays(lb.wl_uniform(1, n, 0.01), None)
        got = {s: n for s, (_, n) in c.profile_read().items()}
        assert got["sort0"] == 1 and got["sort1"] == got["sort3"] == 0
