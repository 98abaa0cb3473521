"""CPU checks of the marching kernels' source: what a wave writes to LDS for the
others is read only after a workgroup barrier, and inline assembly declares the
LDS base register that it writes."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bcm_cgli_amd", "csrc")


def source(name):
    text = open(os.path.join(CSRC, name)).read()
    return re.sub(r"//[^\n]*", "", text)


def block(text, start):
    """The braces that open at or after `start`, with what is between them."""
    a = text.index("{", start)
    depth = 0
    for q in range(a, len(text)):
        depth += {"{": 1, "}": -1}.get(text[q], 0)
        if depth == 0:
            return text[a:q + 1]
    raise AssertionError("unbalanced braces")


@pytest.mark.parametrize("name,loop", [("bcm_flux.hip", "for (int i = i0; i <= i1; ++i)"),
                                       ("bcm_kernels_mixed.hip", "for (int i = start; i <= i1; ++i)")])
def test_norm_sums_of_the_waves_cross_a_barrier(name, loop):
    # Wave 0 adds red[0..3], the sums each wave wrote for a plane.  Between a
    # write and the read of that plane, and between that read and the next
    # plane's write, stands a barrier: taken round the loop, no stretch between
    # two barriers holds both a write and a read.
    body = block(source(name), source(name).index(loop))
    events = [m.lastgroup for m in re.finditer(
        r"(?P<barrier>__syncthreads\(\))|(?P<write>\bred\[[^;=]*\]\s*=(?!=))"
        r"|(?P<read>\bred\[|\bplane_row\(\))", body)]
    assert {"barrier", "write", "read"} <= set(events)
    first = events.index("barrier")
    stretch = set()
    for ev in events[first + 1:] + events[:first + 1]:
        if ev == "barrier":
            assert not {"write", "read"} <= stretch, events
            stretch = set()
        stretch.add(ev)


@pytest.mark.parametrize("name", ["bcm_flux.hip", "bcm_kernels_mixed.hip"])
def test_inline_assembly_declares_m0(name):
    text = source(name)
    writers = 0
    for m in re.finditer(r"asm volatile\((.*?)\);", text, re.S):
        if re.search(r"s_mov_b32 m0", m.group(1)):
            writers += 1
            clobbers = m.group(1).rsplit(":", 1)[1]
            assert '"m0"' in clobbers and '"memory"' in clobbers, m.group(0)
    assert writers
