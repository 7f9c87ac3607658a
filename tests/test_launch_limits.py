"""What the launchers promise the kernels, read from the sources: entry points
run in several host threads, so a kernel's LDS limit is one constant."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quipsharp_amd", "csrc")


def source(name):
    return open(os.path.join(CSRC, name)).read()


FILES = sorted(f for f in os.listdir(CSRC) if "hipFuncAttributeMaxDynamicSharedMemorySize" in source(f))


@pytest.mark.parametrize("name", FILES)
def test_lds_limits_are_constants(name):
    text = source(name)
    for m in re.finditer(r"hipFuncSetAttribute\((.*?),\s*hipFuncAttributeMaxDynamicSharedMemorySize,\s*(.*?)\)\);", text, re.S):
        # a constant, or a limit that a `done` record keeps from being set again or lowered
        guarded = "done" in text[max(0, m.start() - 400):m.start()]
        assert re.fullmatch(r"k[A-Z]\w*", m.group(2)) or guarded, (name, m.group(0))
