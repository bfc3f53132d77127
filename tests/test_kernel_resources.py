"""What the compiler gave the kernels of the built library, where their speed depends on it: registers decide how many
wavefronts a SIMD holds.  Read from the notes of the code objects in liblfhip.so; no GPU needed."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from liteform_ae_amd import _lib

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    blob = open(path, "rb").read()
    at = blob.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        (entries,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(entries):
            offset, size, name = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + name]
            pos += 24 + name
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Name -> (vector registers, bytes of scratch) of every kernel."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    found = {}
    for i, image in enumerate(code_objects(_lib.LIB_PATH)):
        path = tmp_path_factory.mktemp("objects") / f"{i}.elf"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, stdout=subprocess.PIPE, text=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            field = lambda name: re.search(rf"\.{name}:\s+(\S+)", kernel).group(1)  # noqa: E731
            found[field("symbol").strip("'").removesuffix(".kd")] = (int(field("vgpr_count")), int(field("private_segment_fixed_size")))
    return found


def test_plain_csr_product_of_many_features_keeps_three_wavefronts_to_a_simd(kernels):
    """Float features in four pieces of a lane, B inside 4 GB, neither panels nor chunks: 512 registers / 3, in steps of 8."""
    names = [n for n in kernels if "csr_spmm_kernelILi64ELi4EfLb0ELb0E" in n]
    assert len(names) == 1
    registers, scratch = kernels[names[0]]
    assert registers <= 168 and scratch == 0
