"""Register counts of the built kernels, from the metadata of libkate_hip.so's own
code objects: an instantiation that carries steps no plan sends it pays for
their registers with waves per SIMD."""
import os
import re
import struct
import subprocess

import pytest

import kate_amd as K

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(path):
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, data):
        at = m.start() + len(magic)
        count, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(min(count, 8)):
            offset, size, idlen = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + idlen]
            at += 24 + idlen
            if b"gfx950" in name and size:
                yield data[m.start() + offset:m.start() + offset + size]


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """Kernel name (mangled) -> vector registers, accumulators included."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    out, tmp = {}, tmp_path_factory.mktemp("co")
    for i, co in enumerate(code_objects(K.LIB_PATH)):
        path = tmp / f"{i}.co"
        path.write_bytes(co)
        text = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for block in text.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", block).group(1)
            out[name] = int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))
    assert out
    return out


@pytest.mark.parametrize("tile", [10, 11])
def test_complex128_batch_of_wide_gates_keeps_two_waves(registers, tile):
    counts = [v for k, v in registers.items() if re.search(rf"k_batchIdLi{tile}ELi[1-9]ELi4E", k)]
    assert len(counts) == 1 and counts[0] <= 256, counts
