"""Every answer of a launch rule is one that a kernel was built for (CPU only)."""

from __future__ import annotations

import pytest

import launch_rules

ANSWERS = dict(setup_whole_lanes={0, 1}, select_lanes={8, 16, 32}, select_together={0, 1}, geometry_parts={1, 2, 4, 8, 16, 32}, raster_parts={1, 2, 4, 8}, raster_sixteen={0, 1}, gap_waves={4, 8, 16}, sprite_row_parts={1, 4},
               side_stream_pays={0, 1})
MAPS = (1, 2, 100, 160, 161, 320, 511, 512, 513, 899, 900, 1023, 1024, 2000, 4000, 4095, 4096, 4097, 65534)


@pytest.mark.parametrize("rule", launch_rules.RULES)
def test_every_answer_is_one_the_launches_know(rule):
    others = {launch_rules.LINEDEFS: MAPS, launch_rules.BILLBOARDS: (0, 1), launch_rules.NOTHING: (0,)}[launch_rules.RULES[rule]]
    given = {launch_rules.ask(rule, lanes, other) for other in others for lanes in range(1, launch_rules.MOST_LANES + 1)}
    if rule == "select_strips":      # a launch of that many strips' wavefronts, or none
        assert min(given) == 0 and max(given) <= 1024
    else:
        assert given <= ANSWERS[rule]
        assert len(given) > 1, "a rule that always answers alike is none"


def test_strips_of_a_screen_are_shared_in_whole_columns():
    assert all(64 % launch_rules.ask("raster_parts", lanes) == 0 for lanes in range(1, launch_rules.MOST_LANES + 1))
