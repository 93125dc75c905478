"""No kernel of the library keeps data in private memory (per-lane scratch in HBM: a register array or a struct
that the compiler could not split), from the resource notes that the compiler writes beside each kernel."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "endtoend_amd", "lib", "libcccs.so")
LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(fatbin):
    """The gfx950 code objects of an offload bundle section."""
    at = fatbin.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", fatbin, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", fatbin, p)
            if size and b"gfx950" in fatbin[p + 24:p + 24 + ln]:
                yield fatbin[at + off:at + off + size]
            p += 24 + ln
        at = fatbin.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-readelf"), reason="needs ROCm's llvm-readelf")
def test_no_kernel_uses_private_memory(tmp_path):
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={tmp_path}/fatbin", LIB, f"{tmp_path}/copy"],
                   check=True)
    kernels = {}
    for i, co in enumerate(_code_objects((tmp_path / "fatbin").read_bytes())):
        (tmp_path / f"co{i}").write_bytes(co)
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(tmp_path / f"co{i}")], check=True,
                               capture_output=True, text=True).stdout
        names = re.findall(r"^ {4}\.name: +(\S+)", notes, re.M)
        sizes = re.findall(r"^ {4}\.private_segment_fixed_size: +(\d+)", notes, re.M)
        assert len(names) == len(sizes)
        kernels.update(zip(names, map(int, sizes)))
    assert len(kernels) > 40 and any("cone_kernel" in k for k in kernels)
    assert {k: v for k, v in kernels.items() if v} == {}
