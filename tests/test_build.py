"""The native call of kernel objects is an extra: the library is built where it cannot be, and one that was built against
another torch is not used."""

import os
import shutil
import subprocess
import sys
import sysconfig

import pytest
import torch

from tilelang_amd import _lib


def test_library_without_the_native_call(tmp_path):
    csrc = tmp_path / "tilelang_amd" / "csrc"
    os.makedirs(csrc)
    os.makedirs(tmp_path / "include")
    for name in ("Makefile", "host_call.cpp"):
        shutil.copy(os.path.join(_lib.CSRC_DIR, name), csrc)
    shutil.copy(os.path.join(_lib.CSRC_DIR, "..", "..", "include", "dqgemm.h"), tmp_path / "include")
    stale = tmp_path / "tilelang_amd" / ("_hostcall" + sysconfig.get_config_var("EXT_SUFFIX"))
    stale.touch()
    os.utime(stale, (1, 1))
    # no library to build either (a file that stands for it), and an interpreter without torch
    (tmp_path / "tilelang_amd" / "libdqgemm.so").touch()
    proc = subprocess.run(["make", "-C", str(csrc), "all", f"PYTHON={sys.executable} -S", "OBJS="], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "is not built" in proc.stdout and not stale.exists()


@pytest.mark.skipif(_lib.host_call() is None, reason="the native call is not built")
def test_other_torch(monkeypatch):
    monkeypatch.setattr(_lib, "_host_call", None)
    monkeypatch.setattr(torch.version, "git_version", "of another build")
    with pytest.warns(UserWarning, match="built against torch"):
        assert _lib.host_call() is None
    assert _lib.host_call() is None  # said once
    monkeypatch.undo()
    assert _lib.host_call() is not None
