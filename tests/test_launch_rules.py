"""Every answer of a launch rule is one that a kernel was built for (CPU only)."""

from __future__ import annotations

import os
import subprocess
import tempfile

import pytest

import launch_rules

ANSWERS = dict(setup_whole_lanes={0, 1}, select_lanes={8, 16, 32}, select_together={0, 1}, geometry_parts={1, 2, 4, 8, 16, 32}, raster_parts={1, 2, 4, 8}, raster_sixteen={0, 1}, gap_waves={4, 8, 16}, sprite_row_parts={1, 4},
               side_stream_pays={0, 1}, observe_few={0, 1})
MAPS = (1, 2, 100, 128, 129, 160, 161, 279, 280, 320, 399, 400, 511, 512, 513, 659, 660, 899, 900, 1023, 1024, 1699, 1700, 2000, 2299, 2300, 2999, 3000, 4000, 4095, 4096, 4097, 65534)


@pytest.mark.parametrize("rule", launch_rules.RULES)
def test_every_answer_is_one_the_launches_know(rule):
    others = {launch_rules.LINEDEFS: MAPS, launch_rules.BILLBOARDS: (0, 1), launch_rules.NOTHING: (0,)}[launch_rules.RULES[rule]]
    given = {launch_rules.ask(rule, lanes, other) for other in others for lanes in range(1, launch_rules.MOST_LANES + 1)}
    if rule == "select_strips":      # a launch of that many strips' wavefronts, or none
        assert min(given) == 0 and max(given) <= 768
    else:
        assert given <= ANSWERS[rule]
        assert len(given) > 1, "a rule that always answers alike is none"


@pytest.mark.parametrize("rule", ["select_strips", "select_lanes"])
def test_the_selections_rules_change_where_these_maps_are(rule):
    """Every number of linedefs at which an answer changes has one on either side of it in MAPS."""
    given = {linedefs: [launch_rules.ask(rule, lanes, linedefs) for lanes in range(1, launch_rules.MOST_LANES + 1, 16)] for linedefs in range(1, 5001)}
    assert {linedefs for linedefs in range(2, 5001) if given[linedefs] != given[linedefs - 1]} <= {linedefs for linedefs in MAPS if linedefs - 1 in MAPS}


def test_strips_of_a_screen_are_shared_in_whole_columns():
    assert all(64 % launch_rules.ask("raster_parts", lanes) == 0 for lanes in range(1, launch_rules.MOST_LANES + 1))


def test_the_gap_columns_rule_can_be_asked_of_the_lanes_alone():
    """Callers that know no map ask ``gap_waves(lanes)``: a kernel was built for every answer, and small maps' launches follow it as far as they share."""
    source = '#include "gd_rules.h"\n#include <cstdio>\nint main() { for (int n = 1; n <= %d; ++n) printf("%%d ", gap_waves(n)); }\n' % launch_rules.MOST_LANES
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "ask")
        subprocess.run(["g++", "-std=c++17", "-x", "c++", "-I", launch_rules.CSRC, "-o", path, "-"], input=source, text=True, check=True)
        answers = [int(word) for word in subprocess.run([path], capture_output=True, text=True, check=True).stdout.split()]
    assert set(answers) == {8, 16}
    for lanes, answer in enumerate(answers, start=1):
        assert launch_rules.ask("gap_waves", lanes, 600) in (answer, 4)
