"""kmoe_linear_i8: the ctypes mirror of its argument block, and what the host side refuses (no GPU)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L():
    import sys
    sys.path.insert(0, os.path.join(ROOT, "vllm-kunlun_amd"))
    from vllm_kunlun_amd import _lib
    return _lib


def test_layout(L, tmp_path):
    fields = [n for n, _ in L.LinearI8Args._fields_]
    src = tmp_path / "layout.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "kmoe.h"\nint main(void) {\n  printf("%zu", sizeof(kmoe_linear_i8_args));\n'
                   + "".join(f'  printf(" %zu", offsetof(kmoe_linear_i8_args, {f}));\n' for f in fields) + "  return 0;\n}\n")
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    assert out == [C.sizeof(L.LinearI8Args)] + [getattr(L.LinearI8Args, f).offset for f in fields]


def test_refusals(L):
    def call(**over):
        g = L.LinearI8Args()
        for name in ("x", "w", "w_max", "y", "scratch"):
            setattr(g, name, 4096)
        g.rows, g.n, g.k, g.ld_x, g.ldy, g.w_layout = 3, 64, 128, 128, 64, L.KMOE_W_TILED
        g.scratch_bytes = L.lib.kmoe_linear_i8_workspace_bytes(3, 128)
        for name, value in over.items():
            setattr(g, name, value)
        return L.lib.kmoe_linear_i8(g, None)
    assert L.lib.kmoe_linear_i8_workspace_bytes(3, 128) == 512 + 12
    for over, rc in (({"x": 0}, -1), ({"scratch": 0}, -1), ({"n": 24}, -2), ({"k": 72}, -2), ({"rows": -1}, -2), ({"k": 65552}, -2),
                     ({"scratch_bytes": 500}, -4), ({"scratch": 4100}, -4), ({"w_layout": L.KMOE_W_ROWMAJOR}, -3),
                     ({"ld_x": 120}, -2), ({"ld_x": 132}, -2), ({"ldy": 62}, -2), ({"ldy": 60}, -2), ({"w": 4104}, -2),
                     ({"y": 4100}, -2), ({"act_dtype": 7}, -3)):
        assert call(**over) == rc, over
    assert call(rows=0, scratch_bytes=0) == 0
    far = 0xfff00000 // 65536  # codes beyond 32-bit offsets: only through lod
    assert call(rows=far, k=65536, ld_x=65536, scratch_bytes=1 << 40) == -2 and b"32-bit" in L.lib.kmoe_last_error()
