"""Work-group memory and the barriers of a kernel's loops, read from the kernel sources (CPU only).

Between the last barrier of a loop's body and the first one of its next round nothing keeps the wavefronts of a work-group
apart: one may have begun the next round while another still reads what the last round left in LDS.  No loop may therefore write
a ``__shared__`` variable before its first barrier that it reads after its last.
"""

from __future__ import annotations

import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "env-gradoom-turbo-torch_amd", "csrc")
BARRIER = re.compile(r"__syncthreads(?:_or|_and|_count)?\s*\(")


def _closing(text: str, start: int) -> int:
    """Index of the bracket that closes the one at ``start``."""

    pairs = {"(": ")", "{": "}"}
    opening, depth = text[start], 0
    for at in range(start, len(text)):
        depth += (text[at] == opening) - (text[at] == pairs[opening])
        if depth == 0:
            return at
    raise AssertionError("unbalanced brackets")


def _loops(body: str):
    """Bodies of the loops of a kernel, the inner ones too, their conditions included."""

    for match in re.finditer(r"\b(?:for|while)\s*\(|\bdo\s*\{", body):
        start = match.end() - 1
        if body[start] == "(":
            end = _closing(body, start)
            brace = re.match(r"\s*\{", body[end + 1 :])
            if brace is None:
                continue
            start = end + brace.end()
        yield body[start + 1 : _closing(body, start)]


def unordered_writes(source: str) -> list[tuple[str, str]]:
    """(kernel, variable) of every ``__shared__`` variable that a loop writes before its first barrier and reads after its last."""

    source = re.sub(r"/\*.*?\*/|//[^\n]*", "", source, flags=re.S)
    found = []
    for match in re.finditer(r"__global__[^;{]*?\b(\w+)\s*\((?!\()[^;{]*\{", source):
        start = match.end() - 1
        header = source[match.start() : start]
        kernel = [name for name in re.findall(r"\b(\w+_kernel)\s*\(", header)][-1]
        body = source[start + 1 : _closing(source, start)]
        declared = re.sub(r"\[[^\]]*\]", "", " , ".join(re.findall(r"__shared__\s+([^;]+);", body)))
        names = {re.findall(r"\w+", part)[-1] for part in declared.split(",") if re.findall(r"\w+", part)}
        for loop in _loops(body):
            barriers = list(BARRIER.finditer(loop))
            if not barriers:
                continue
            # what a barrier's condition reads is read before it
            before, after = loop[: barriers[0].start()], loop[_closing(loop, barriers[-1].end() - 1) :]
            for name in sorted(names):
                written = re.search(rf"\b{name}\b\s*(?:\[[^=;]*\])?(?:\.\w+)?\s*[-+|&^]?=(?!=)", before) or re.search(rf"atomic\w+\(\s*&?{name}\b", before)
                if written and re.search(rf"\b{name}\b", after):
                    found.append((kernel, name))
    return found


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.hip"))), ids=os.path.basename)
def test_no_loop_overwrites_what_its_last_round_still_reads(path):
    with open(path) as handle:
        assert unordered_writes(handle.read()) == []


@pytest.mark.parametrize("head, expected", [
    ("bits[tid] = 0; __syncthreads();", [("walk_kernel", "bits")]),
    ("__syncthreads(); bits[tid] = 0;", []),
    ("if (!__syncthreads_or(bits[tid])) break;", []),
    ("atomicOr(&bits[tid], 1); __syncthreads();", [("walk_kernel", "bits")]),
])
def test_the_reading_finds_a_write_before_the_barrier(head, expected):
    kernel = """
    __global__ void __launch_bounds__(256) walk_kernel(int rounds, int *out) {   // bits[0] = 1;
        __shared__ int bits[256];
        for (int k = 0; k < rounds; ++k) { %s __syncthreads(); while (out[k]) { out[k] += bits[k]; } }
    }
    """ % head
    assert unordered_writes(kernel) == expected
