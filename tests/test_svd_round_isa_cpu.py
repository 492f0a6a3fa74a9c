"""The Jacobi round kernels' order of the converged flag and the Gram's first
loads, in the gfx950 code object (compiled here, CPU only).

A captured run keeps launching rounds over converged problems: its kernels
(FIRST) test the flag, word 1 of the problem's flags, and branch before any
vector load of four words (X), so that such a round moves nothing."""
import os
import re
import subprocess

import pytest

from conftest import ROOT
from test_isa_cpu import HIPCC, _kernel_body

SRC = os.path.join(ROOT, "tenet.jl_amd", "csrc", "k_svd.hip")
FLAG_TEST = re.compile(r"s_load_dword (s\d+), s\[\d+:\d+\], 0x4\n"  # the flag
                       r"(?:(?!.*s_cmp).*\n)*?\s+s_cmp_\w+ \1, 0\n"  # compared
                       r"(?:(?!.*s_cmp).*\n)*?\s+s_cbranch_scc")  # and branched on


@pytest.fixture(scope="module")
def isa(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("isa") / "k_svd.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", SRC, "-o", str(out)], check=True,
                   capture_output=True, cwd=os.path.dirname(SRC))
    return out.read_text()


@pytest.mark.parametrize("alone,units", [(1, 1), (0, 1), (1, 0)])
def test_captured_rounds_test_the_flag_before_loading(isa, alone, units):
    body = _kernel_body(isa, f"_ZN5tenet21svd_round_mfma_kernelILb{alone}ELb{units}ELb1EEEvNS_8SvdBatchEii")
    before = body[:re.search(r"(flat|global|buffer)_load_dwordx4", body).start()]
    assert FLAG_TEST.search(before)
