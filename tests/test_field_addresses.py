"""The sensor kernels address a node by its plane (64 bits, one value for a
workgroup) and a 32-bit byte offset in the plane.  Both parts are computed on
the host here, from the header the kernels use, and must add up to the node's
element in the field: an explicit upwind box without the filter has no limit of
505 cells an axis, and from 4 GiB a field (810^3 cells fit the card) an offset
of 32 bits alone wraps onto other planes."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include "geo.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv)
{
    const int n[3] = {atoi(argv[1]), atoi(argv[2]), atoi(argv[3])};
    long pi, pj, pk;
    const astr::Geo g = astr::padded_geo(n, pi, pj, pk);
    printf("%ld\n", pi * pj * pk);
    for (int e = 0; e < 27; ++e) {
        const int i = e % 3 * n[0] / 2, j = e / 3 % 3 * n[1] / 2, k = e / 9 * n[2] / 2;
        printf("%d %d %d %ld %ld %u\n", i, j, k, astr::gidx(g, i, j, k), astr::plane_elem(g, k),
               astr::plane_byte(g, i, j));
    }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    inc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
    if not cxx or not os.path.isdir(inc):
        pytest.skip("needs g++ and the HIP headers")
    d = tmp_path_factory.mktemp("addr")
    (d / "addr.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w", "-I" + inc,
                    "-I" + os.path.join(ROOT, "astr_gpu_amd", "csrc"), "-o", str(d / "addr"),
                    str(d / "addr.cpp")], check=True)
    return str(d / "addr")


@pytest.mark.parametrize("dims", [(16, 16, 16), (33, 17, 20), (1024, 1025, 0), (505, 505, 505),
                                  (810, 810, 810), (1000000, 16, 40), (16, 40, 1000000),
                                  (17, 200000, 30)])
def test_plane_and_offset(program, dims):
    out = subprocess.run([program, *map(str, dims)], check=True, capture_output=True, text=True)
    lines = out.stdout.split("\n")
    nfield = int(lines[0])
    pi = (16 + dims[0] + 1 + 5 + 15) // 16 * 16
    pj = dims[1] + 11
    assert nfield == pi * pj * (dims[2] + 11)
    for ln in lines[1:28]:
        i, j, k, elem, plane, off = map(int, ln.split())
        assert elem == 16 + i + pi * (j + 5 + pj * (k + 5)) < nfield
        assert off % 8 == 0 and plane + off // 8 == elem, (i, j, k)
    if dims == (810, 810, 810):
        assert 8 * nfield > 2 ** 32  # the last node's whole offset takes more than 32 bits
