"""The parts of bench.py that follow the sources and the library's dispatch."""
from __future__ import annotations

import os
import sys

from conftest import PKG_NAME, ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_the_stamped_conv_finds_its_markers():
    """--hconv-phases builds a copy of csrc/hconv.hip with a stamp at each phase of the
    256-pixel kernel: every marker is there once, and the other kernels have none."""
    src = open(os.path.join(ROOT, PKG_NAME, "csrc", "hconv.hip")).read()
    out = bench.hconv_stamped_source(src)
    assert out.count("HCP(") - out.count("#define HCP(") == 5 and "g_hcp[4096 * 128]" in out
    at = out.index("void hconv_fp8_kernel(")
    kernel = out[at:out.index("\n}\n", at)]
    assert kernel.count("HCP(") == 5
    assert out.replace(kernel, "").count("HCP(") == 1      # its definition
