"""Which levels the LDS-tiled stencil kernels serve (ael::tiles_serve), on the
CPU: a halo load takes any component of a field through one base and a 32-bit
byte offset, so the last value of a three-component FP64 field has to lie below
2^32 bytes; boxes of the sizes in use stay tiled."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "stencil_lds.h"
int main(int argc, char** argv) {
    for (int q = 1; q + 2 < argc; q += 3) {
        ael::Lvl L{};
        L.nx = std::atoi(argv[q]);
        L.ny = std::atoi(argv[q + 1]);
        L.nz = std::atoi(argv[q + 2]);
        L.N = (long)L.nx * L.ny * L.nz;
        std::printf("%d\\n", (int)ael::tiles_serve(L));
    }
    return 0;
}
"""

# nodes; the limit lies at 178,956,970 nodes: 563^3 is below it, 564^3 above, and
# 2^32 / 24 = 178,956,970.67 between the last two
SHAPES = [(33, 65, 65), (34, 34, 34), (129, 129, 129), (257, 257, 257), (513, 513, 513), (563, 563, 563),
          (564, 564, 564), (641, 641, 641), (769, 769, 641), (803, 803, 803), (1281, 513, 257), (1025, 513, 345),
          (65, 65, 42356), (65, 65, 42357)]


def test_tiles_serve_fields_within_32_bit_offsets(tmp_path):
    from alamo_amd import build
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not found")
    src = tmp_path / "limits.hip"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "limits")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", build.CSRC, "-o", exe, str(src)], check=True,
                   timeout=300)
    args = [str(n) for shape in SHAPES for n in shape]
    out = subprocess.run([exe, *args], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    for (nx, ny, nz), tiled in zip(SHAPES, out):
        last = 8 * (3 * nx * ny * nz - 1)  # byte offset of the last value of an FP64 field
        want = min(nx, ny, nz) >= 34 and last + 8 < 2 ** 32
        assert int(tiled) == int(want), (nx, ny, nz)
        if int(tiled):
            assert last == last % 2 ** 32
