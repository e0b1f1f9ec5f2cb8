"""The launch plan of ckv_attention_active, walked on the CPU (tests/native/attention_plan_walk.cpp):
for every combination of KV heads 1-256, groups 1-16, both head sizes, query and cache lengths around
the plan's limits and workspaces from none to plenty, the plan's kernel form exists, its splits fit
and its work items are each taken once."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_every_plan_can_be_launched(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "attention_plan_walk"
    subprocess.run([gxx, "-O2", "-std=c++17", f"-I{ROOT / 'chunkkv_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "attention_plan_walk.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300).stdout
    checked, bad = map(int, out.splitlines()[-1].split())
    assert checked > 1_000_000 and bad == 0, out
