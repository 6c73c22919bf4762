"""What the launch code of the kernels keeps to, read from its sources."""

import os
import re

import pytest

from fei_amd.ops import build


@pytest.mark.parametrize("name", build.SOURCES + build.HEADERS)
def test_no_state_of_the_process(name):
    """No static variable but constants: what a launch has told one device says
    nothing of the next, and another thread may launch meanwhile."""
    with open(os.path.join(build.CSRC, name)) as f:
        code = re.sub(r"//[^\n]*", "", f.read())
    found = [m.group(0) for m in re.finditer(
        r"\bstatic\b(?!\s+(?:constexpr|const|inline|_*device_*|_*host_*))"
        r"[^;{(]*[;=]", code)]
    assert not found
