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


@pytest.mark.parametrize("name,kernel", [("qs_linear_wide.hip", "wg_kernel"), ("qs_linear_wide.hip", "wp_kernel"),
                                         ("qs_linear_fused.hip", "linear_fused_kernel"),
                                         ("qs_linear_batched.hip", "bm_kernel")])
def test_kernels_with_tables_at_lds_address_0_refuse_static_lds(name, kernel):
    """lds_word reads the code tables at their LDS addresses: static LDS would
    come first and move them, so the launcher asks the runtime for it."""
    text = source(name)
    at = text.index("LaunchKernelGGL(" + ("" if kernel == "wp_kernel" else "(") + kernel)
    before = text[max(0, at - 2000):at]
    launcher = before[max(before.rfind("\nint "), before.rfind("\ntemplate <")):]
    if "sharedSizeBytes == 0" not in launcher:  # in a helper that the launcher calls with the kernel
        helper = re.search(r"(\w+)\(\(const void\*\)" + kernel, launcher)
        assert helper, (name, kernel)
        body = text[text.index("int " + helper.group(1) + "("):]
        launcher = body[:body.index("\n}")]
    assert "sharedSizeBytes == 0" in launcher, (name, kernel)
