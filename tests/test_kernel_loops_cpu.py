"""Loops that count their requests under way (s_waitcnt vmcnt) hold no spilled register: its reload waits for all of them.  Read from the built library."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "vyomai_amd", "lib", "libvyom_hip.so")
BIN = "/opt/rocm/llvm/bin/"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """The gfx950 code object of every source."""
    data = open(LIB, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 24)


def scratch_in_loops(listing):
    """Addresses of scratch accesses between a backward branch and its target."""
    lines = [(int(m[2], 16), m[1].strip()) for m in re.finditer(r"^\t(.*?)// ([0-9A-F]+):", listing, re.M)]
    loops = []
    for at, text in lines:
        m = re.match(r"s_c?branch\S* (\d+)", text)
        if m:
            jump = int(m[1])
            to = at + 4 + 4 * (jump - 65536 if jump >= 32768 else jump)
            if to <= at:
                loops.append((to, at))
    assert lines
    return [(hex(at), text) for at, text in lines if text.startswith("scratch_") and any(a <= at <= b for a, b in loops)], loops


@pytest.mark.parametrize("kernels", ["attn_bwd_dq_kernel", "attn_bwd_dkdv_kernel", "wgrad_tn_bf16_rows_kernel", "gemm_nt_bf16_m16_kernel"])
def test_no_scratch_in_loops(kernels, tmp_path):
    assert os.path.exists(LIB)
    seen = 0
    for i, obj in enumerate(code_objects()):
        if kernels.encode() not in obj:
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        names = subprocess.run([BIN + "llvm-objdump", "-t", str(path)], capture_output=True, text=True, check=True).stdout
        names = sorted({line.split()[-1] for line in names.splitlines() if re.search(r" F \.text", line) and kernels in line})
        for name in names:
            listing = subprocess.run([BIN + "llvm-objdump", "-d", "--disassemble-symbols=" + name, str(path)], capture_output=True, text=True,
                                     check=True).stdout
            found, loops = scratch_in_loops(listing)
            assert loops and not found, (name, found)
            seen += 1
    assert seen
