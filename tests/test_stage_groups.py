"""The row groups a small block's stage goes in (row_groups, pga_stagecore.hpp) on the CPU: they take every row
once, and their grid keeps to the 65 535 a box's planes keep to."""

import ctypes
import subprocess

import pytest

from peregrine_amd import build

SOURCE = """
#include "pga_internal.hpp"
#include "pga_stagecore.hpp"
using namespace pga;
extern "C" void groups(int n0, int n1, int n2, int kc, int ne, int *out) {
  StageArgs a{};
  a.n0 = n0, a.n1 = n1, a.n2 = n2;
  row_groups(a, ne, (n2 + kc - 1) / kc);
  out[0] = a.groups, out[1] = a.rows;
}
"""


@pytest.fixture(scope="module")
def groups(tmp_path_factory):
    d = tmp_path_factory.mktemp("groups")
    (d / "groups.hip").write_text(SOURCE)
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", f"-I{build.CSRC}", "-shared",
                    str(d / "groups.hip"), "-o", str(d / "groups.so")], check=True, capture_output=True)
    return ctypes.CDLL(str(d / "groups.so")).groups


@pytest.mark.parametrize("ne", [5, 9, 13, 20])
def test_a_stage_s_grid_keeps_to_its_limits(groups, ne):
    out = (ctypes.c_int * 2)()
    for n0, n1 in ((1, 1), (2, 1), (3, 3), (61, 47), (1000, 1000)):
        for n2 in (1, 2, 33, 1000, 3276, 3277, 5041, 5042, 7282, 13107, 32767, 32768, 65535):
            for kc in (1, 2, 7):
                groups(n0, n1, n2, kc, ne, out)
                n, rows = out
                assert n * -(-n2 // kc) <= 65535
                assert n >= 1 and (n - 1) * rows < ne <= n * rows
    groups(61, 47, 33, 1, ne, out)
    assert out[0] > 1
