"""Launch-shape rules that results do not show (no GPU needed): common.hpp's
functions, compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "common.hpp"
#include <cstdio>
using namespace rv;
int main()
{
    // a batch's launch of a kind goes by the kind's cells, whichever member is
    // first: 27 cells of Nq = 8 and six members of 2744
    const int64_t all = 27 + 6 * 2744;
    std::printf("%d %d %d ", kind_waves(3, 8, LAW_EULER, 8, all, 0), kind_waves(3, 8, LAW_EULER, 4, all, 0),
                kind_waves(2, 8, LAW_ADVECTION, 8, all, 0));
    std::printf("%d %d ", kind_waves(3, 8, LAW_ADVECTION, 8, all, 0), kind_waves(3, 8, LAW_ADVECTION, 8, 27, 0));
    // ... unless the first member's was chosen
    std::printf("%d %d ", kind_waves(3, 8, LAW_EULER, 8, all, 4), kind_waves(3, 8, LAW_EULER, 4, 27, 2));
    // an operator alone: both sides of 1024 waves (Nq = 4: four cells a wave)
    std::printf("%d %d %d %d ", default_waves(3, 8, 8, 1024, true), default_waves(3, 8, 8, 1025, true),
                default_waves(3, 4, 4, 4096, true), default_waves(3, 4, 4, 4097, true));
    std::printf("%d\n", default_waves(3, 8, 8, 32768, false));
}
"""


def test_waves_per_workgroup(tmp_path):
    src, exe = tmp_path / "shape.cpp", tmp_path / "shape"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "raven.jl_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert out.split() == "1 2 1 2 1 4 2 1 4 1 2 1".split()
