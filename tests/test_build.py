"""The part of the build that depends on the installed torch: compile and link options taken from an interpreter."""
import importlib.util
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def make(tmp_path):
    """`make` on a copy of the makefile alone, with an interpreter that prints `says` or, with None, fails."""
    csrc = tmp_path / "csrc"
    csrc.mkdir()
    shutil.copy(os.path.join(ROOT, "trl_amd", "csrc", "Makefile"), csrc)
    python = tmp_path / "some python"
    options = csrc / "build" / "torch.mk"

    def run(goal, says):
        python.write_text("#!/bin/sh\n" + ("echo half; exit 1\n" if says is None else f"echo '{says}'\n"))
        python.chmod(0o755)
        done = subprocess.run(["make", "-C", str(csrc), goal, f"PYTHON={python}"], capture_output=True, text=True, timeout=60)
        return done.returncode, (options.read_text().strip() if options.exists() else None)

    run.options = options
    return run


def test_options_of_torch_follow_the_interpreter(make):
    rc, options = make("build/torch.mk", None)
    assert rc != 0 and options is None  # (an interpreter without torch leaves nothing that the next run takes as good)
    assert make("build/torch.mk", "TORCH_CXX := -Done") == (0, "TORCH_CXX := -Done")
    before = os.stat(make.options).st_mtime_ns
    assert make("build/torch.mk", "TORCH_CXX := -Done")[0] == 0
    assert os.stat(make.options).st_mtime_ns == before  # (the same torch: nothing is compiled again)
    assert make("build/torch.mk", "TORCH_CXX := -Dtwo") == (0, "TORCH_CXX := -Dtwo")
    rc, options = make("build/torch.mk", None)
    assert rc != 0 and options == "TORCH_CXX := -Dtwo"
    assert make("clean", None)[0] == 0  # (needs no torch)


def test_build_uses_the_running_interpreter(monkeypatch):
    spec = importlib.util.spec_from_file_location("_trl_amd_build", os.path.join(ROOT, "trl_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    commands = []
    monkeypatch.setattr(build.subprocess, "run", lambda command, **kwargs: commands.append(command))
    monkeypatch.setattr(build.os.path, "exists", lambda path: True)
    build.build(clean=False)
    assert commands and all(f"PYTHON={sys.executable}" in c for c in commands if "asan" not in c)
