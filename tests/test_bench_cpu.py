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


def test_kernel_names_are_the_library_s():
    """The kernels that a bench line names: tiles that a few images do not fill, strips of large
    batches and one-tap products with few rows, where a rule on widths and channels alone errs."""
    names = bench.library_kernels
    assert names(128, 32, 32, 128, 128, 3, 1, 1) == (
        "hconv_fp8_kernel", "hconv_fp8_kernel", "hwgrad_partial_kernel<32, false>")
    assert names(128, 16, 16, 256, 256, 3, 1, 1)[2] == "hwgrad_partial_kernel<16, false>"
    assert names(32, 64, 64, 128, 128, 3, 1, 1)[2] == "hwgrad_partial_kernel<32, true>"
    assert names(1, 64, 64, 128, 128, 3, 1, 1)[2] == "wgrad_partial_kernel"
    assert names(57, 9, 40, 256, 256, 3, 1, 1)[2] == "hwgrad_partial_kernel<8, true>"
    assert names(128, 32, 32, 128, 128, 3, 2, 1) == (
        "igemm_fp8_kernel", "igemm_fp8_kernel", "wgrad_partial_kernel")
    assert names(128, 16, 16, 512, 256, 1, 1, 0)[0] == "onetap_fp8_kernel"
    assert names(1, 8, 8, 512, 256, 1, 1, 0)[0] == "igemm_fp8_kernel"      # 2 tiles of 256 CUs
    assert names(32768, 1, 1, 768, 256, 1, 1, 0)[:2] == ("igemm_fp8_kernel", "onetap_fp8_kernel")
    # every conv workload of the bench takes its names from there, and the profile's byte counts
    # are kept under them
    import json
    traffic = json.load(open(bench.PROFILE_TRAFFIC))["cfg2"]
    assert names(128, 32, 32, 128, 128, 3, 1, 1)[2] + "+wgrad_reduce_kernel" in traffic
