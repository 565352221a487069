"""The rule that gives a small system the one-launch sort (sort_one_limit)."""
import ctypes


# where one launch and four measured the same, by the steps between re-sorts:
# one launch was ahead at the first size and behind at the second
def test_limit_lies_between_the_sizes_measured(engine):
    limit = ctypes.CDLL(engine.library_path())._ZN4mdpd14sort_one_limitEi
    for period, ahead, behind in [(1, 2000, 5000), (2, 3500, 7000), (3, 5000, 9000), (4, 7000, 10240)]:
        assert ahead <= limit(period) < behind, period
    got = [limit(p) for p in (-5, 0, 1, 2, 3, 4, 5, 6, 1000, 2**31 - 1)]
    assert got == sorted(got) and got[0] == limit(1) and got[-1] == 10240
