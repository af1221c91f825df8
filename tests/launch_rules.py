"""The rules by which a frame's launches are cut (``csrc/gd_rules.h``), compiled for the host: where each changes its answer."""

from __future__ import annotations

import ctypes as C
import functools
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "env-gradoom-turbo-torch_amd", "csrc")
MOST_LANES = 4096        # of one chunk: larger batches are rendered chunk by chunk

# what a rule is asked beside the lanes: the map's linedefs, or whether there are billboards
LINEDEFS, BILLBOARDS, NOTHING = "linedefs", "billboards", None
RULES = dict(setup_whole_lanes=LINEDEFS, select_strips=LINEDEFS, select_lanes=LINEDEFS, select_together=NOTHING, geometry_parts=NOTHING, raster_parts=NOTHING, raster_sixteen=NOTHING, gap_waves=LINEDEFS,
             sprite_row_parts=NOTHING, side_stream_pays=BILLBOARDS, observe_few=NOTHING)


@functools.lru_cache(maxsize=1)
def library() -> C.CDLL:
    source = ['#include "gd_rules.h"'] + [
        f'extern "C" int ask_{name}(int lanes, int other) {{ (void)other; return (int){name}({"lanes" if asked is NOTHING else "lanes, other"}); }}'
        for name, asked in RULES.items()
    ]
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "librules.so")
        subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-x", "c++", "-I", CSRC, "-o", path, "-"], input="\n".join(source) + "\n", text=True, check=True)
        return C.CDLL(path)


def ask(rule: str, lanes: int, other: int = 0) -> int:
    return getattr(library(), "ask_" + rule)(lanes, int(other))


def lines(rule: str, other: int = 0) -> list[int]:
    """The batch sizes from which on the rule's answer is another than that for one lane less."""

    return [lanes for lanes in range(2, MOST_LANES + 1) if ask(rule, lanes, other) != ask(rule, lanes - 1, other)]
