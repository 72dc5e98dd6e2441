"""LVX_LIB names the library every operator runs, the native ones included."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import os, sys
sys.path.insert(0, sys.argv[1])
import torch
from lv_xattn import _lib
o, lse, ws = _lib.host().forward_buffers(torch.zeros(1, 8, 16, 128, dtype=torch.bfloat16), 16, 4, False)    # asks the library
assert ws.numel() == _lib.load().lvx_fwd_workspace_bytes(_lib.AttnShape(1, 8, 2, 128, 16, 64, 1, 1.0), 16, 4)
print(sorted({line.split()[-1] for line in open("/proc/self/maps") if "liblvx" in line}))
"""


def test_one_library_is_mapped_and_it_is_the_named_one(tmp_path):
    from lv_xattn import _lib
    _lib.load()
    named = str(tmp_path / "liblvx_other.so")
    shutil.copy(_lib.LIB_PATH, named)
    r = subprocess.run([sys.executable, "-c", PROGRAM, os.path.join(ROOT, "lv-xattn_amd")], env=dict(os.environ, LVX_LIB=named),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip().splitlines()[-1] == str([named])


def test_a_library_of_another_version_is_refused(monkeypatch, tmp_path):
    """An older build lacks functions this package calls; its version says so."""
    from lv_xattn import _lib
    header = open(os.path.join(ROOT, "include", "lvx.h")).read()
    assert _lib.VERSION == int(re.search(r"^#define\s+LVX_VERSION\s+(\d+)", header, re.M).group(1))
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    (tmp_path / "old.c").write_text("int lvx_version(void) { return 103; }")
    subprocess.run([gcc, "-shared", "-fPIC", "-o", str(tmp_path / "old.so"), str(tmp_path / "old.c")], check=True)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "old.so"))
    with pytest.raises(_lib.LvxError, match="version 103"):
        _lib.load()
