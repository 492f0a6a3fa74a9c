"""How many workgroups share the rows of one matrix's Jacobi pairs (host rule,
compiled here): dealt over the XCDs, a pair's on one of them, they never exceed
an XCD's CUs, as long as one workgroup a pair does not."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = """
#include <cstdio>
#include "internal.h"
int main() {
  for (long long pairs = 1; pairs <= 300; ++pairs)
    for (long long strips = 1; strips <= 130; strips += 3)
      std::printf("%lld %lld %lld\\n", pairs, strips, (long long)tenet::svd_row_shares(pairs, strips));
}
"""


def test_shares_fit_an_xcd(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "shares.cpp", tmp_path / "shares"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "tenet.jl_amd", "csrc"), str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    rows = [tuple(map(int, x.split())) for x in subprocess.run([str(exe)], check=True, capture_output=True,
                                                               text=True).stdout.splitlines()]
    assert len(rows) == 300 * 44
    for pairs, strips, q in rows:
        on_one_xcd = -(-pairs // 8)
        assert q >= 1 and (q == 1 or on_one_xcd * q <= 32), (pairs, strips, q)
        assert q == 1 or q <= -(-strips // 4)
        # no share is left out that both limits allow
        assert q + 1 > max(1, min(32 // on_one_xcd, -(-strips // 4)))
