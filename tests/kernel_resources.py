"""Registers, spills and LDS of the kernels in the built library, from the
metadata notes of its gfx950 code objects."""
import os
import re
import shutil
import struct
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "taichi_elements_amd", "csrc")
_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(_MAGIC)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(_MAGIC))
        p = at + len(_MAGIC) + 8
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + name_len]
            p += 24 + name_len
            if b"gfx950" in name:
                yield data[at + offset:at + offset + size]
        at = data.find(_MAGIC, at + 1)


def kernel_resources():
    """{demangled kernel name without its arguments: dict of vgprs, spills, lds}"""
    from taichi_elements_amd import build
    readelf = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
    if not (os.path.exists(build.LIB) and os.path.exists(readelf) and shutil.which("c++filt")):
        pytest.skip("needs the built library, llvm-readelf and c++filt")
    found = {}
    with open(build.LIB, "rb") as f:
        data = f.read()
    for obj in _code_objects(data):
        with tempfile.NamedTemporaryFile(suffix=".elf") as f:
            f.write(obj)
            f.flush()
            notes = subprocess.run([readelf, "--notes", f.name], capture_output=True, text=True,
                                   check=True).stdout
        for entry in notes.split("  - .agpr_count:")[1:]:
            def field(key):
                return re.search(rf"\n    \.{key}:\s+(\S+)", entry).group(1)
            found[field("name")] = dict(vgprs=int(field("vgpr_count")),
                                        spills=int(field("vgpr_spill_count")),
                                        lds=int(field("group_segment_fixed_size")))
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    return {n.split("(")[0].replace("void ", "").replace("mpm::", ""): r
            for n, r in zip(names, found.values())}


def workgroups_per_cu(res):
    """Workgroups of 256 threads (a wave per SIMD) of a kernel that a gfx950 CU
    holds: 512 registers a lane and SIMD, given out eight at a time, at most
    eight waves a SIMD, 160 KiB of LDS."""
    registers = 512 // max(8, -(-res["vgprs"] // 8) * 8)
    lds = (160 * 1024) // max(res["lds"], 1)
    return min(registers, 8, lds)


def constant(name):
    """Value of a constexpr int of the kernel sources."""
    for header in ("mpm_kernels.h", "mpm_kernels.hip", "mpm_device.h"):
        with open(os.path.join(CSRC, header)) as f:
            m = re.search(rf"constexpr int [^;]*\b{name} = ([^,;]+)", f.read())
        if m:
            return eval(m.group(1), {"__builtins__": {}})  # integer arithmetic
    raise KeyError(name)
