"""What the compiler recorded about the kernels it put into the library, read from the kernels' own metadata (no GPU)."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(path, tmp_path):
    """(mangled name, metadata text) of every gfx950 kernel in a library's offload bundles."""
    blob = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + n].decode()
            pos += 24 + n
            if "gfx950" in triple and size:
                code = tmp_path / "code.elf"
                code.write_bytes(blob[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(code)], capture_output=True, text=True, check=True).stdout
                for block in notes.split("- .agpr_count")[1:]:
                    yield re.search(r"\.symbol:\s+(\S+)\.kd", block).group(1), block
        at = blob.find(magic, at + 1)


@pytest.mark.skipif(not os.path.exists(READELF), reason="the ROCm toolchain's llvm-readelf is not installed")
def test_no_kernel_spills_vector_registers(tmp_path):
    """A spilled register is a trip through memory in the innermost loop (fp16 backward with SiLU and 20-67 of them: 1.3 to
    3 times the time)."""
    from causal_conv1d import _lib
    spilled, seen = {}, set()
    for name, block in kernels(_lib.LIB_PATH, tmp_path):
        seen.add(re.match(r"_ZN5canon\d+(canon_\w+_kernel)", name).group(1))
        n = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", block).group(1))
        if n:
            spilled[name] = n
    assert not spilled
    assert {"canon_bwd_blc_kernel", "canon_bwd_bcl_kernel", "canon_bwd_bcl_short_kernel", "canon_fwd_blc_kernel"} <= seen
