"""The multiply-adds with a row broadcast are written as instructions, so the
compiler sees one operation: an accumulator must not share a register with an
operand that a later instruction of the block still reads, also where both
start with the same value.  Read from the code compiled for gfx950 (no GPU).
"""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "suzerain_amd", "csrc")

# accumulators that hold u's (one row) and u's and l's (four rows) values
SOURCE = r"""
#include "sz_row.hpp"
template <typename R> __global__ void one(R *p)
{
    p += threadIdx.x;
    const R lx = p[0], ly = p[64], ux = p[128], uy = p[192];
    R ax = ux, ay = uy;
    sz::fnms_row1<3>(ax, ay, lx, ly, ux, uy);
    p[0] = ax;
    p[64] = ay;
}
template <typename R> __global__ void four(R *p)
{
    p += threadIdx.x;
    const R lx = p[0], ly = p[64], ux = p[128], uy = p[192];
    R a[8] = {ux, uy, p[256], p[320], p[384], p[448], lx, ly};
    sz::fnms_row4<4>(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], lx, ly, ux, uy);
    for (int i = 0; i < 8; ++i) p[64 * i] = a[i];
}
template __global__ void one<double>(double *);
template __global__ void one<float>(float *);
template __global__ void four<double>(double *);
template __global__ void four<float>(float *);
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    """The instructions (destination, sources) of each block of assembly."""
    d = tmp_path_factory.mktemp("row")
    src, out = d / "row.hip", d / "row.s"
    src.write_text(SOURCE)
    subprocess.run(["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-I", CSRC,
                    "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", str(src), "-o",
                    str(out)], check=True, capture_output=True)
    found = []
    for text in re.findall(r"ASMSTART(.*?)ASMEND", out.read_text(), re.S):
        ops = re.findall(r"v_fmac_f(?:32|64)_dpp (\S+), (\S+), (\S+) row_newbcast", text)
        found.append([(d_, {a.lstrip("-"), b.lstrip("-")}) for d_, a, b in ops])
    return [b for b in found if b]


def test_accumulators_have_registers_of_their_own(blocks):
    assert sorted(len(b) for b in blocks) == [4, 4, 16, 16]
    for ops in blocks:
        written = {d for d, _ in ops}
        read = set().union(*(s for _, s in ops))
        assert not written & read, (written & read, ops)
