"""Registers of the built kernels, from the code objects in libdsx.so (no GPU needed)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from ds_splat_amd import _native

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))


def kernels(tmp_path):
    """{mangled name: its metadata's numbers} of every kernel in the library."""
    data, found = open(_native.LIB_PATH, "rb").read(), {}
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, data):
        at = m.end()
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + length].decode()
            at += 24 + length
            if "gfx950" in name and size:
                part = tmp_path / "code.elf"
                part.write_bytes(data[m.start() + offset:m.start() + offset + size])
                notes = subprocess.run([READELF, "--notes", str(part)], capture_output=True, text=True, check=True).stdout
                for one in notes.split("  - .agpr_count:")[1:]:
                    found[re.search(r"\.name: +(\S+)", one).group(1)] = {
                        k: int(v) for k, v in re.findall(r"\.(\w+): +(\d+)\n", one)}
    return found


@pytest.mark.skipif(READELF is None, reason="needs llvm-readelf")
def test_the_blend_backward_keeps_everything_in_registers(tmp_path):
    """A value that is spilled and read back in a round of the walk waits for all of the last round's adds to memory."""
    walks = {k: v for k, v in kernels(tmp_path).items() if re.search(r"\d+blend_bwd_\w*kernel", k)}
    assert len(walks) == 5, sorted(walks)
    assert {k: v["vgpr_spill_count"] for k, v in walks.items() if v["vgpr_spill_count"]} == {}
