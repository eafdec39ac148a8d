"""The attend's split-K rules (host logic, no GPU): the fused step's rule (partials merged in-kernel) and the standalone
attend's (merged by the combine kernel) pick the partition counts that were fastest on MI355X at the measured shapes
(32K with S = 1092 and 128K with S = 4164, B = 1..16, h = 1, 2, 4); the docstring of merged_partitions holds the
timings, where the rule is within 0.4 us of the best P per layer."""
from __future__ import annotations

import pytest

from attention_lab.hip_attend import merged_partitions, one_launch_step, sparse_partitions, step_partitions


@pytest.mark.parametrize("BG,S,h,want", [
    (8, 1092, 1, 8), (8, 1092, 2, 8), (8, 1092, 4, 8),
    (16, 1092, 1, 8), (16, 1092, 2, 8), (16, 1092, 4, 8),
    (32, 1092, 1, 8), (32, 1092, 4, 4),
    (64, 1092, 1, 4), (64, 1092, 2, 4), (64, 1092, 4, 2),
    (128, 1092, 1, 2), (128, 1092, 2, 2), (128, 1092, 4, 1),
    (8, 4164, 2, 16), (8, 4164, 4, 8), (16, 4164, 4, 8), (32, 4164, 2, 8), (32, 4164, 4, 4),
])
def test_merged_rule_picks_the_measured_best(BG, S, h, want):
    assert merged_partitions(BG, S, h) == want == sparse_partitions(BG, S, h, merged=True)


def test_short_lists_are_not_split_below_128_rows_and_the_combine_rule_is_unchanged():
    assert merged_partitions(8, 132, 2) == 1 and merged_partitions(8, 300, 2) == 2
    # the standalone attend (combine kernel): B=1 P=8, B=16 h=4 P=1 (two head groups), B=16 h=1 P=1
    assert sparse_partitions(8, 1092, 2) == 8 and sparse_partitions(128, 1092, 4) == 1 and sparse_partitions(128, 1092, 1) == 1


@pytest.mark.parametrize("h", [1, 2, 4, 8])
def test_merged_rule_never_asks_for_a_second_round(h):
    """Every batch and row count: at most 256 workgroups (one round, a workgroup fills a CU) wherever the (b, g) rows
    alone allow it, and no partition without rows."""
    for BG in range(1, 300):
        for S in (1, 68, 127, 132, 300, 447, 448, 454, 1092, 4164, 9000):
            P = merged_partitions(BG, S, h)
            assert 1 <= P <= max(1, min(16, S // 56))
            assert P == 1 or BG * P <= 256


@pytest.mark.parametrize("BG,S,h,want", [
    (24, 1092, 4, 8), (40, 1092, 4, 4), (56, 1092, 4, 3), (96, 1092, 4, 2), (24, 4164, 4, 8), (24, 5068, 4, 8),
    (96, 454, 4, 2), (8, 324, 8, 1), (24, 1092, 8, 4), (16, 454, 8, 1),
])
def test_steps_of_separate_launches_keep_the_grid_their_attend_was_measured_with(BG, S, h, want):
    """A step whose rows are returned, or past what one launch selects and attends: at four heads per KV group the attend's
    small workgroups want more partitions than one round of the one-launch kernel's, at eight longer ones; other h as
    there."""
    assert merged_partitions(BG, S, h, one_launch=False) == want != merged_partitions(BG, S, h)
    for other in (1, 2, 3, 5, 6, 7):
        assert merged_partitions(BG, S, other, one_launch=False) == merged_partitions(BG, S, other)


def test_which_steps_run_in_one_launch():
    assert one_launch_step(4, 32700, False) and one_launch_step(1, 131072, False)
    assert not one_launch_step(4, 32700, True) and not one_launch_step(4, 131073, False)
    assert not any(one_launch_step(h, 32700, False) for h in (3, 5, 6, 7, 8))
    assert step_partitions(96, 1092, 4, 32700, 1024, False) == 1 and step_partitions(96, 1092, 4, 32700, 1024, True) == 2
    assert step_partitions(96, 1092, 4, 0, 0, False) == sparse_partitions(96, 1092, 4)
