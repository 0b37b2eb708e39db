"""No kernel of the library keeps anything in scratch memory: the metadata of
the GPU code object built into it."""
import os
import re
import struct
import subprocess

import pytest

import pixelforge_amd as pf

LLVM = "/opt/rocm/llvm/bin"


def _kernels(tmp_path):
    """Kernel name -> bytes of scratch memory per lane."""
    objcopy, readelf = os.path.join(LLVM, "llvm-objcopy"), os.path.join(LLVM, "llvm-readelf")
    if not (os.path.exists(objcopy) and os.path.exists(readelf)):
        pytest.skip("no LLVM tools")
    fat = tmp_path / "fatbin"
    subprocess.run([objcopy, "-O", "binary", "--only-section=.hip_fatbin", pf.LIB_PATH, str(fat)], check=True)
    data = fat.read_bytes()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    out, at = {}, data.find(magic)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in target:
                elf = tmp_path / "code.o"
                elf.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([readelf, "--notes", str(elf)], check=True, capture_output=True, text=True).stdout
                for block in re.split(r"\n\s+- \.agpr_count|\n\s+- \.args", notes):
                    name = re.search(r"^\s+\.name:\s+(_Z\w+|\w+)\s*$", block, re.M)
                    size_ = re.search(r"\.private_segment_fixed_size:\s+(\d+)", block)
                    if name and size_:
                        out[re.findall(r"\.symbol:\s+'?(\w+)", block)[-1]] = int(size_.group(1))
        at = data.find(magic, at + 1)
    return out


def test_no_kernel_uses_scratch_memory(tmp_path):
    kernels = _kernels(tmp_path)
    assert len(kernels) > 100
    assert not {k: v for k, v in kernels.items() if v}
