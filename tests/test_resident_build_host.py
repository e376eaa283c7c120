"""What the compiler made of the chip-resident time loop's kernels, read from
the built library's own code objects (gfx950); no device is involved."""
import os
import re
import struct
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "..", "denise-black-edition_amd", "libdnhip.so")
LLVM = "/opt/rocm/llvm/bin/"
NAME = re.compile(r"k_resident" + r"ILi(\d+)" + r"ELi(\d+)" * 6 + "E")


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The code objects that hold kernels of the loop."""
    tmp = tmp_path_factory.mktemp("code_objects")
    fat = tmp / "fat"
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", LIB, "/dev/null"], check=True)
    data = fat.read_bytes()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    found = []
    for at in (m.start() for m in re.finditer(magic, data)):
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, pos - 8)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n]
            pos += 24 + n
            code = data[at + off:at + off + size]
            if b"gfx950" in name and b"k_resident" in code:
                found.append(tmp / f"{len(found)}.co")
                found[-1].write_bytes(code)
    assert len(found) == 18  # six operator lengths, three groups of physics
    return found


def test_no_flat_instructions(objects):
    """Every access says which memory it means: FLAT ones find out from an
    aperture kept in registers."""
    for path in objects:
        text = subprocess.run([LLVM + "llvm-objdump", "-d", str(path)], capture_output=True, text=True, check=True).stdout
        assert "k_resident" in text and "global_load" in text
        assert "flat_" not in text


def instances(objects):
    """(half-order, rows, columns, pitch, physics, mechanisms, direction): vector registers spilled"""
    out = {}
    for path in objects:
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(path)], capture_output=True, text=True,
                               check=True).stdout
        for block in notes.split("  - .agpr_count:")[1:]:
            key = tuple(map(int, NAME.search(re.search(r"\.name:\s+(\S+)", block).group(1)).groups()))
            out[key] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", block).group(1))
    return out


def test_spilled_registers(objects):
    """No kernel with several rows per thread spills 100 registers or more,
    but for the two of order 8 that the GPU tests run."""
    got = instances(objects)
    assert len({k[0] for k in got}) == 6 and len({(k[4], k[5], k[6]) for k in got}) == 16
    heavy = {k: n for k, n in got.items() if k[1] > 1 and n >= 100}
    assert set(heavy) <= {(4, 3, 4, 72, 1, 2, 0), (4, 3, 4, 72, 4, 0, 1)}, heavy
    assert max(got.values()) < 168, max(got.items(), key=lambda kv: kv[1])
