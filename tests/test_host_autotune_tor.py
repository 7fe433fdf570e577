"""The torontonian's schedule choice: only mode counts that have both walks decide."""
from gbskernels_amd import autotune


def t(dfs, bfs, grouped=9.0):
    return {"dfs": dfs, "bfs": bfs, "grouped": grouped}


def test_counts_with_one_kernel_do_not_decide():
    both = {3: t(2.0, 1.0), 4: t(2.0, 1.0), 5: t(2.0, 1.0)}
    # two timings of one kernel, "breadth-first" slower by noise
    for slow in (6, 8, 20):
        assert autotune.choose_tor({**both, slow: t(1.0, 1.2)}, 0.02) == (0, 32)
        assert autotune.choose_tor({**both, slow: {"bfs": 1.2, "grouped": 2.0}}, 0.02) == (0, 32)


def test_counts_with_both_walks_decide():
    assert autotune.choose_tor({3: t(2.0, 1.0), 4: t(1.0, 1.5), 5: t(2.0, 1.0), 8: t(1.0, 1.0)}, 0.02) == (0, 3)
    assert autotune.choose_tor({3: t(1.0, 1.01), 4: t(1.0, 1.5)}, 0.02) == (0, 3)
    assert autotune.choose_tor({2: t(1.0, 1.5), 3: t(2.0, 1.0)}, 0.02) == (0, 0)


def test_grouped_kernel_needs_a_clear_gain_at_every_step():
    times = {2: t(1.0, 1.0, 0.5), 4: t(1.0, 1.0, 0.5), 6: {"bfs": 1.0, "grouped": 0.99}}
    assert autotune.choose_tor(times, 0.02)[0] == 4
