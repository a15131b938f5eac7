"""What the compiled kernels' own metadata says, read from the library that was built here.  No GPU needed."""
import os
import re
import struct
import subprocess

import pytest

from ratchet_amd import _lib, build

READELF = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """the gfx950 code objects inside the library, one per source: after the magic a count, then (offset, size, length of the
    name, name) of each entry"""
    blob = open(_lib.LIB_PATH, "rb").read()
    at = blob.find(MAGIC)
    while at >= 0:
        (count,), pos = struct.unpack_from("<Q", blob, at + len(MAGIC)), at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if "gfx950" in name and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + 1)


@pytest.mark.parametrize("softmax, least", [("softmax16_stream_kernel", 100), ("softmax16_row_kernel", 40)])
def test_the_softmax_table_lies_at_the_start_of_lds(tmp_path, softmax, least):
    """the kernel reads its table at LDS address 0 + 2 * bits, where its dynamic LDS starts only as long as nothing
    that is compiled into the kernel declares static LDS of its own"""
    seen = 0
    for k, code in enumerate(code_objects()):
        path = tmp_path / ("%d.co" % k)
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s+- \.(?:agpr_count|args)", notes):
            name = re.search(r"\.name:\s+(\S+)", kernel)
            if name and softmax in name.group(1):
                seen += 1
                assert re.search(r"\.group_segment_fixed_size:\s+0\n", kernel), name.group(1)
    assert seen >= least, seen
