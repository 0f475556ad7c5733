"""Kernels that end at once when a solve's stop flag is set and that may set it
themselves: their workgroups read it once, for all wavefronts.  A return by
wavefront before a barrier would leave the others with a sum that lacks its
part.  Checked on the sources."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ngsolve_amd", "csrc")
SETS = re.compile(r"->done = |CheckResidual\(|DirectionBeta\(|ctl\[0\] = |MultiCgHead\(")
RETURNS = re.compile(r"if \((stop(_flag)? && \*stop(_flag)?|S->done|ctl\[0\])\) return")


def kernels(name):
    """(name, body) of every kernel of a source file; the branches that only
    kernels without the setting code compile are taken out."""
    text = open(os.path.join(CSRC, name)).read()
    for m in re.finditer(r"__global__ (?:__launch_bounds__\([^()]*\) )?void (\w+)\(", text):
        at = text.index("{", m.end())
        depth, end = 1, at + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        yield m.group(1), re.sub(r"} else {\n    if \(stop_flag && \*stop_flag\) return;", "", text[at:end])


@pytest.mark.parametrize("name", ["cg.hip", "spmv.hip", "multicg.hip"])
def test_setters_read_the_flag_once(name):
    setters = [(k, b) for k, b in kernels(name) if SETS.search(b)]
    assert setters
    for k, body in setters:
        if "__syncthreads" not in body and not re.search(r"SumPartials|StorePartial|DirectionBeta", body):
            continue  # no barrier: nothing is shared between its wavefronts
        assert not RETURNS.search(body), k
