"""The ctypes ``tsattn_step_desc`` against the header as gcc lays it out."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

from tensorsmith_hip import _lib

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc unavailable")
def test_step_desc_layout_matches_header(tmp_path):
    names = [f[0] for f in _lib.StepDesc._fields_]
    src = tmp_path / "step.c"
    src.write_text('#include <stddef.h>\n#include <stdio.h>\n#include "tsattn.h"\nint main(void){\n'
                   'printf("%zu\\n", sizeof(tsattn_step_desc));\n'
                   + "".join(f'printf("%zu\\n", offsetof(tsattn_step_desc, {n}));\n' for n in names)
                   + "return 0;}\n")
    exe = tmp_path / "step"
    subprocess.run(["gcc", "-I", str(ROOT / "include"), str(src), "-o", str(exe)], check=True)
    got = [int(x) for x in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]
    assert got == [ctypes.sizeof(_lib.StepDesc)] + [getattr(_lib.StepDesc, n).offset for n in names]


def test_step_refuses_without_launching():
    lib = _lib.load()
    desc = _lib.StepDesc()
    assert lib.tsattn_cached_step_workspace(desc) == 0
    assert lib.tsattn_cached_step(desc, None, 0, None) == _lib.ERR_INVALID
