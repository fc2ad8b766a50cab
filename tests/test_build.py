"""When the native host module is compiled again (no compiler runs here)."""

import importlib.util
import os
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def build(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("ck_build", os.path.join(ROOT, "cute-kernels_amd", "build.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    module.runs = 0
    for name, file in (("HOST_PATH", "host.so"), ("HOST_SOURCE", "host.cpp"), ("OBJ_DIR", "objects")):
        monkeypatch.setattr(module, name, str(tmp_path / file))
    (tmp_path / "host.cpp").write_text("")
    monkeypatch.setattr(module, "INCLUDE", str(tmp_path))
    (tmp_path / "ck_mi355.h").write_text("")

    def run(command, **kwargs):
        module.runs += 1
        (tmp_path / "host.so").write_text("")
        return subprocess.CompletedProcess(command, 0, "", "")

    monkeypatch.setattr(module.subprocess, "run", run)
    return module


def test_host_module_is_compiled_once(build):
    build.build_host()
    build.build_host()
    assert build.runs == 1
    build.build_host(force=True)
    assert build.runs == 2


@pytest.mark.parametrize("changed", ["source", "torch", "flags"])
def test_host_module_is_compiled_again(build, monkeypatch, changed):
    build.build_host()
    if changed == "source":
        later = os.path.getmtime(build.HOST_PATH) + 10
        os.utime(build.HOST_SOURCE, (later, later))
    elif changed == "torch":
        monkeypatch.setattr(torch, "__version__", "99.0")
    else:
        command = build._host_command
        monkeypatch.setattr(build, "_host_command", lambda output: command(output) + ["-DOTHER"])
    build.build_host()
    assert build.runs == 2
