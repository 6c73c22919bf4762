"""What the launch code of the kernels keeps to, read from its sources."""

import os
import re
import shutil
import subprocess

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


@pytest.mark.parametrize("name", ["attn_prefill.hip", "tile.hip"])
def test_m0_is_only_used_by_the_loads_that_set_it(name, tmp_path):
    """load_lds_from sets m0 and cannot tell the compiler, whose own uses would find
    another value: there are none in these files."""
    if shutil.which(build.HIPCC) is None:
        pytest.skip("needs hipcc")
    src = os.path.join(build.CSRC, name)
    with open(src) as f:
        assert "load_lds_from" in f.read()
    out = tmp_path / "device.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", src,
                    "-o", str(out)], check=True, capture_output=True, timeout=600)
    asm = out.read_text()
    assert re.search(r"\bs_mov_b32 m0\b", asm)
    own = re.sub(r"#ASMSTART.*?#ASMEND", "", asm, flags=re.S)
    assert not re.search(r"\bm0\b", own)
    # nobody else has such loads
    for other in build.SOURCES:
        with open(os.path.join(build.CSRC, other)) as f:
            assert (other in ("attn_prefill.hip", "tile.hip")
                    or "load_lds_from" not in f.read())
