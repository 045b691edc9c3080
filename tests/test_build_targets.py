"""What `make` builds by itself, and slimkernels_amd._lib.build() with it: the C library, and the native host side of the torch
calls exactly where torch has GPU support."""
import os
import shutil
import subprocess

import pytest

from slimkernels_amd import _lib

CSRC = os.path.dirname(_lib.LIB_PATH)
pytestmark = pytest.mark.skipif(shutil.which("make") is None, reason="needs make")


def _dry_run(*args):
    run = subprocess.run(["make", "-n", "-B", "-C", CSRC, *args], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stderr
    return run.stdout


@pytest.mark.parametrize("gpu", [True, False])
def test_default_target(tmp_path, gpu):
    os.makedirs(tmp_path / "lib")
    if gpu:
        (tmp_path / "lib" / "libc10_hip.so").write_text("")
    out = _dry_run(f"TORCH={tmp_path}")
    assert "-o libslimk_w2a8.so" in out and ("-o ../torch/_native.so" in out) == gpu


def test_without_torch():
    out = _dry_run("TORCH=")
    assert "-o libslimk_w2a8.so" in out and "_native" not in out


@pytest.mark.parametrize("gpu", [True, False])
def test_build_function(monkeypatch, tmp_path, gpu):
    """The command of build() is that of the default target."""
    os.makedirs(tmp_path / "lib")
    if gpu:
        (tmp_path / "lib" / "libc10_hip.so").write_text("")
    commands = []
    monkeypatch.setattr(_lib.subprocess, "run", lambda cmd, **kw: commands.append(cmd))
    assert _lib.build() == _lib.LIB_PATH
    monkeypatch.undo()
    assert len(commands) == 1 and commands[0][0] == "make"
    run = subprocess.run([*commands[0], "-n", f"TORCH={tmp_path}"], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stderr
    assert "-o libslimk_w2a8.so" in run.stdout and ("-o ../torch/_native.so" in run.stdout) == gpu
