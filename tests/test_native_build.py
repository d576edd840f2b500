"""The build of the native libraries (``loqa_hub_amd/_native/build.py``), without compiling."""
import importlib.util
import subprocess

import pytest

from loqa_hub_amd._native import build


@pytest.fixture
def no_compiler(monkeypatch, tmp_path):
    """Libraries are written nowhere; commands are noted and taken as done."""
    ran = []

    def run(cmd, **kw):
        ran.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(subprocess, "run", run)
    return ran


def test_without_torch_the_other_libraries_are_built(no_compiler, monkeypatch):
    monkeypatch.setattr(importlib.util, "find_spec", lambda name: None)
    assert [p.rsplit("/", 1)[1] for p in build.build(only=("libloqa_runtime.so", "libloqa_launch.so"))] == ["libloqa_runtime.so"]


@pytest.mark.parametrize("abi", [False, True])
def test_the_module_has_the_abi_of_torch(no_compiler, monkeypatch, abi):
    import torch
    monkeypatch.setattr(torch, "compiled_with_cxx11_abi", lambda: abi)
    assert build.build(only=("libloqa_launch.so",))
    assert f"-D_GLIBCXX_USE_CXX11_ABI={int(abi)}" in no_compiler[-1]
    assert len(no_compiler) == 1 and build.build(only=("libloqa_launch.so",)) and len(no_compiler) == 1      # up to date
