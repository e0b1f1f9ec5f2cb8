"""bench.py's argument checks, before it touches a device."""

import os
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_concurrent_prefills_are_switched_off():
    """Several HipEngine prefills from several host threads stalled on the GPU, cause not found: asking
    for that measurement is an error that says so."""
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")
    r = subprocess.run([sys.executable, "bench.py", "--workload", "replay", "--concurrent-ttft"], cwd=ROOT, env=env,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2 and "stalled" in r.stderr and "cause not found" in r.stderr, (r.returncode, r.stderr)
