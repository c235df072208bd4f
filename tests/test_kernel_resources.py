"""What the built kernels need at launch, from the metadata of the library's own
code objects.

No kernel may need scratch memory: the runtime allocates it when such a kernel is
launched, and aborts the queue where the device's memory is taken, as it is beside
pools that keep what they were given until an allocation fails."""

import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """The gfx950 ELF images bundled in the library, one for each source file."""
    import compas_amd

    data = open(compas_amd.library_path(), "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name and size > 0:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    path = tmp_path_factory.mktemp("objects") / "object"
    out = {}
    for image in code_objects():
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for size, symbol in re.findall(r"\.private_segment_fixed_size:\s+(\d+).*?\.symbol:\s+(\S+)", notes, re.S):
            out[symbol] = int(size)
    return out


def test_no_kernel_needs_scratch(kernels):
    assert any("pssfp_map" in k for k in kernels) and any("fisp_real" in k for k in kernels)
    assert {k: v for k, v in kernels.items() if v} == {}
