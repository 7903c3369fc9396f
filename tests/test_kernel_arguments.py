"""Metadata of the built gfx950 kernels.

The one-patch work table (SegSingleT) travels by value.  No kernel keeps a copy
of it in private memory, where every read of the patch would be a scratch load
and its address no constant memory."""
import os
import struct
import subprocess

import pytest
import yaml

from hamers_amd.build import HIPCC, LIB

READELF = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(image):
    at = image.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", image, at + len(MAGIC))
        o = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", image, o)
            target = image[o + 24:o + 24 + length].decode()
            o += 24 + length
            if "gfx950" in target and size:
                yield image[at + offset:at + offset + size]
        at = image.find(MAGIC, at + len(MAGIC))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    with open(LIB, "rb") as f:
        image = f.read()
    out = []
    for i, obj in enumerate(_code_objects(image)):
        path = tmp_path_factory.mktemp("code") / f"{i}.o"
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        doc = notes[notes.index("---"):]
        doc = doc[:doc.index("\n...")]
        out += yaml.load(doc, Loader=getattr(yaml, "CSafeLoader", yaml.SafeLoader))["amdhsa.kernels"]
    assert out
    return [k for k in out if "10SegSingleT" in k[".name"]]


def test_no_private_copy_of_the_one_patch_table(kernels):
    assert kernels and all(k[".args"][0][".value_kind"] == "by_value" for k in kernels)
    copies = [k[".name"] for k in kernels if k[".private_segment_fixed_size"] >= k[".args"][0][".size"]]
    assert not copies, f"{len(copies)} kernels, {copies[0]}"
