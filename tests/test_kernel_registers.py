"""Registers of the built kernels, on the CPU: the sweeps of the tiled stencil
kernels, periodic ones included, are held to so many waves a SIMD that nothing
spills to scratch memory (the compiler's own counts, from the code objects of the
built library).  Not asked of the periodic FP64 Fapply and residual, which spill
two registers at 3 waves a SIMD and are faster so than at 2 without."""
import os
import re
import struct
import subprocess

import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(path, tmp):
    """The gfx950 code objects of a library, written to files."""
    data = open(path, "rb").read()
    out = []
    for m in re.finditer(MAGIC, data):
        at = m.start() + len(MAGIC)
        n, = struct.unpack_from("<Q", data, at)
        at += 8
        if n > 64:
            continue
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + idlen]
            at += 24 + idlen
            if b"gfx950" in name and size:
                f = tmp / f"{len(out)}.co"
                f.write_bytes(data[m.start() + off:m.start() + off + size])
                out.append(str(f))
    return out


def test_tiled_sweeps_do_not_spill(tmp_path):
    from alamo_amd import elastic
    if not os.path.exists(elastic.LIB_PATH) or not os.path.exists(READELF):
        pytest.skip("libalamo_elastic.so not built, or llvm-readelf absent")
    spills = {}
    for co in code_objects(elastic.LIB_PATH, tmp_path):
        text = subprocess.run([READELF, "--notes", co], capture_output=True, text=True, check=True).stdout
        # one metadata map per kernel, its keys in alphabetical order
        pairs = re.findall(r"\.name:\s+(_Z\S+)(?:(?!\.name:).)*?\.vgpr_spill_count:\s+(\d+)", text, flags=re.S)
        spills.update((n, int(s)) for n, s in pairs)
    tiled = {n: s for n, s in spills.items() if "k_stencil_lds" in n or "k_stencil_iso" in n}
    assert len(tiled) >= 40, sorted(spills)[:5]
    # template arguments after the tile: T = d or f, OP = Li2E
    sweeps = {n: s for n, s in tiled.items() if re.search(r"EE[df]Li2E", n)}
    assert len(sweeps) == 16, sorted(sweeps)  # lds: 2 types x 3 layouts of C x periodic or not; iso: 2 x 2
    assert all(s == 0 for s in sweeps.values()), {n: s for n, s in sweeps.items() if s}
