"""Register use of the built decode kernels: the walks stream K and V at the
rate of HBM, and an instance whose registers spill adds scratch accesses to
every tile of every wave."""
import re
import shutil
import struct
import subprocess

import pytest

from cvsa.ops import _lib

READELF = shutil.which("llvm-readelf") or shutil.which("/opt/rocm/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 code objects of the library's offload bundles."""
    for m in re.finditer(MAGIC, data):
        at = m.start()
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, name_len = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + name_len]
            entry += 24 + name_len
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]


@pytest.mark.skipif(READELF is None, reason="needs llvm-readelf")
def test_decode_kernels_use_no_scratch(tmp_path):
    seen, spilled = 0, []
    for obj in _code_objects(_lib.LIB_PATH.read_bytes()):
        path = tmp_path / "code.o"
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True,
                               check=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            if not re.search("listed_decode|listed_append|score_spec|streamk_decode", name):
                continue
            seen += 1
            if any(int(re.search(rf"\.{key}:\s+(\d+)", kernel)[1])
                   for key in ("private_segment_fixed_size", "vgpr_spill_count")):
                spilled.append(name)
    # Four kernels per group size 1 to 16 at the least.
    assert seen >= 64
    assert not spilled
