"""Workgroups of the single-launch decode step that start late (the device is
shared): the code the kernel runs at their start and at the step's end
(qwen3-iree_amd/csrc/step_roles.h), compiled with g++ into a program that lets
them start at any point of a step's end."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_late_workgroups_keep_the_steps_role(tmp_path):
    exe = tmp_path / "step_roles_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror",
                    f"-I{REPO / 'qwen3-iree_amd' / 'csrc'}",
                    str(REPO / "tests" / "native" / "step_roles_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok")
