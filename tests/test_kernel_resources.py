"""Registers of the kernels built here, from the metadata of the library's
code objects: the wavefronts per SIMD that the batch's walks are meant to run
with (512 vector registers per SIMD lane, handed out in eights)."""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from massivemds_amd import build as hipbuild

READELF = Path("/opt/rocm/lib/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

pytestmark = pytest.mark.skipif(not READELF.exists() or shutil.which("c++filt") is None,
                                reason="llvm-readelf or c++filt absent")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled name up to its arguments: (vector registers, spilled ones, scratch bytes)}"""
    if not hipbuild.LIB.exists():
        hipbuild.build()
    data = hipbuild.LIB.read_bytes()
    out = {}
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if "gfx950" not in target or size == 0:
                continue
            path = tmp_path_factory.mktemp("code") / "object"
            path.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([str(READELF), "--notes", str(path)], capture_output=True, text=True, check=True)
            for block in re.split(r"\n  - \.agpr_count|\n  - \.args", notes.stdout)[1:]:
                name = re.search(r"\.name: +(\S+)", re.sub(r"\n +- .*?(?=\n    \.)", "", block, flags=re.S))
                values = [re.search(rf"\n    \.{key}: +(\d+)", block)
                          for key in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size")]
                if name and all(values):
                    out[name.group(1)] = tuple(int(v.group(1)) for v in values)
        at = data.find(MAGIC, at + 1)
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True, check=True).stdout
    return {re.sub(r"^void mdship::|\(.*", "", n): v for n, v in zip(names.splitlines(), out.values())}


def _waves(registers):
    return min(8, 512 // (-(-registers // 8) * 8))


# wavefronts per SIMD by kernel dimension, truncated symmetric data: FP32; FP64
# with plain additions (3), with grouped ones (7) and either, looked up per item
# (19: up to four dimensions, larger ones are launched apart)
@pytest.mark.parametrize("real,flags,waves", [
    ("float", 3, {1: 6, 2: 5, 3: 5, 4: 4, 5: 4, 6: 4, 8: 3, 10: 2}),
    ("double", 3, {1: 6, 2: 5, 3: 5, 4: 4, 5: 4, 6: 4, 8: 3, 10: 3}),
    ("double", 7, {1: 5, 2: 4, 3: 4, 4: 4, 5: 4, 6: 3, 8: 3, 10: 2}),
    ("double", 19, {1: 5, 2: 4, 3: 4, 4: 4})])
def test_batch_walks_keep_their_wavefronts(kernels, real, flags, waves):
    for p, w in waves.items():
        registers, _, _ = kernels[f"batch_tile_kernel<{real}, {p}, {flags}>"]
        assert _waves(registers) >= w, (p, registers)


def test_no_walk_spills(kernels):
    walks = {n: v for n, v in kernels.items() if re.match(r"batch_tile_kernel|tile_kernel|row_delta_kernel", n)}
    assert len(walks) > 300
    assert not [n for n, (_, spilled, scratch) in walks.items() if spilled or scratch]
