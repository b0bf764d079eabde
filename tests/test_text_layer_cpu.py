"""The ctypes mirror of vy_text_layer against a C compiler, and the entry point's argument checks."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_struct_mirror(tmp_path):
    from vyomai_amd._lib import VyTextLayer as T
    src = '#include "vyom_hip.h"\n#include <stdio.h>\n#include <stddef.h>\nint main(void) { printf("%zu", sizeof(vy_text_layer));\n' + \
          "".join(f'printf(" %zu", offsetof(vy_text_layer, {f[0]}));\n' for f in T._fields_) + "return 0; }\n"
    c, exe = tmp_path / "t.c", tmp_path / "t"
    c.write_text(src)
    subprocess.check_call(["gcc", "-I", os.path.join(ROOT, "include"), str(c), "-o", str(exe)])
    got = [int(v) for v in subprocess.check_output([str(exe)], text=True).split()]
    assert got == [ctypes.sizeof(T)] + [getattr(T, f[0]).offset for f in T._fields_]


def test_argument_checks():
    from vyomai_amd import _lib
    with pytest.raises(_lib.VyomHipError, match="null operand"):
        _lib.call("vy_text_layer_fwd", None, None, None, 1, 1, None, 0, None)
    buf = (ctypes.c_char * 256)()
    p = ctypes.addressof(buf)
    l = _lib.VyTextLayer(h=2, hk=2, dh=64, ffn=512, dtype=_lib.VY_BF16)
    with pytest.raises(_lib.VyomHipError, match="workspace too small"):
        _lib.call("vy_text_layer_fwd", ctypes.addressof(l), p, p, 1, 8, p, 256, None)
    l.mask_kind = _lib.MASK_ADDITIVE
    with pytest.raises(_lib.VyomHipError, match="bad sizes or mask"):
        _lib.call("vy_text_layer_fwd", ctypes.addressof(l), p, p, 1, 8, p, 256, None)
