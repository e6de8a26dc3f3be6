"""Vector registers of the built step kernels: the instantiation that most replicas run leaves
room for as many waves per SIMD as its launches were measured with."""
import pathlib
import re
import shutil
import struct
import subprocess

import pytest

import tild

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def _vgprs(tmp):
    """Kernel name -> vector registers, of every gfx950 code object in the library."""
    lib, magic, out, pos = tild.LIB_PATH.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (start := lib.find(magic, pos)) >= 0:
        (n,), at = struct.unpack_from("<Q", lib, start + 24), start + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", lib, at)
            target, at = lib[at + 24:at + 24 + length], at + 24 + length
            if b"gfx950" in target and size:
                co = tmp / "code_object"
                co.write_bytes(lib[start + off:start + off + size])
                notes = subprocess.run([READELF, "--notes", str(co)], capture_output=True, text=True, check=True).stdout
                for k in notes.split("  - .")[1:]:
                    name, v = re.search(r"\.name:\s+(_Z\S+)", k), re.search(r"\.vgpr_count:\s+(\d+)", k)
                    if name and v:
                        out[name.group(1)] = int(v.group(1))
        pos = start + 24
    return out


# 512 registers per SIMD lane: 128 are four waves, 84 six
@pytest.mark.parametrize("kernel,limit", [("k_grad_reg", 128), ("k_c2r_reg", 128), ("k_tile_depositILi512ELi1ELb0E", 84)])
def test_the_lean_instantiation_keeps_its_waves(kernel, limit, tmp_path):
    if not pathlib.Path(READELF).exists():
        pytest.skip("no llvm-readelf")
    v = [r for name, r in _vgprs(tmp_path).items() if kernel in name]
    assert v and min(v) <= limit, v
