"""The staged faces' tiles (face_tiles, pga_flux.hpp) on the CPU: whatever the box and the species count, a
launch asks for no more LDS than any launch may (64 KB), and its tiles hold every face's stencil."""

import ctypes
import subprocess

import pytest

from peregrine_amd import build

SOURCE = """
#include "pga_flux.hpp"
using namespace pga;
extern "C" long long tile_bytes(int axis, int e0, int e1, int e2, int ns, long long *faces) {
  const Box3 b{0, 0, 0, e0, e1, e2};
  const FaceTiles t = face_tiles(axis, b, ns);
  *faces = face_tile_count(t) * (axis ? FLAT : t.shape);
  return (long long)sizeof(double) * face_tile_slots(t) * slot_doubles(ns);
}
"""


@pytest.fixture(scope="module")
def tile_bytes(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "tiles.hip").write_text(SOURCE)
    lib = d / "tiles.so"
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", f"-I{build.CSRC}", "-shared", str(d / "tiles.hip"),
                    "-o", str(lib)], check=True, capture_output=True)
    fn = ctypes.CDLL(str(lib)).tile_bytes
    fn.restype = ctypes.c_longlong
    return fn


def test_no_tile_passes_a_launch_s_lds(tile_bytes):
    faces = ctypes.c_longlong()
    for axis in range(3):
        for e0 in (1, 2, 15, 16, 17, 32, 33, 49, 63, 64, 65, 128, 1000):
            for e1 in (1, 2, 8, 9, 12, 13, 16, 64, 65):
                for e2 in (1, 4, 8, 9, 64, 65):
                    for ns in (1, 2, 9, 12, 13, 14, 15, 16):
                        n = tile_bytes(axis, e0, e1, e2, ns, ctypes.byref(faces))
                        assert 0 < n <= 65536, (axis, e0, e1, e2, ns, n)
                        assert faces.value >= e0 * e1 * e2
