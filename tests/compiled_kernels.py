"""What the compiler reports of the kernels inside libmi355_moe.so (registers, scratch), read without a GPU."""
import functools
import os
import re
import struct
import subprocess
import tempfile

from therock_amd import _lib

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def tools_there():
    return os.path.exists(os.path.join(LLVM, "llvm-readelf"))


def code_objects():
    """One ELF image per translation unit with kernels."""
    data = open(_lib.LIB_PATH, "rb").read()
    images = []
    for at in (m.start() for m in re.finditer(re.escape(MAGIC), data)):
        count = struct.unpack_from("<Q", data, at + len(MAGIC))[0]
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + name_len].decode()
            pos += 24 + name_len
            if "gfx950" in name and size:
                images.append(data[at + offset:at + offset + size])
    return images


def notes(image):
    with tempfile.NamedTemporaryFile() as f:
        f.write(image)
        f.flush()
        return subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", f.name], check=True, stdout=subprocess.PIPE, text=True).stdout


@functools.lru_cache(maxsize=None)
def kernels():
    """{mangled name: what its code object's notes say of it}"""
    got = {}
    for image in code_objects():
        for block in re.split(r"\n\s+- \.agpr_count", notes(image))[1:]:
            said = dict(re.findall(r"^\s+\.(symbol|private_segment_fixed_size|vgpr_count|vgpr_spill_count):\s+(\S+)", block, re.M))
            name = said.pop("symbol").removesuffix(".kd")
            got[name] = {k: int(v) for k, v in said.items()}
    return got
