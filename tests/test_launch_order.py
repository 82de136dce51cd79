"""CPU check of the longest-first launch order (tests/cpp/check_launch_order.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_launch_order_serves_every_unit_once(tmp_path):
    exe = tmp_path / "check_launch_order"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    f"-I{ROOT / 'chia_proj_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "check_launch_order.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and "0 violations" in out.stdout, out.stdout + out.stderr
    planted = subprocess.run([str(exe), "planted"], capture_output=True, text=True)
    assert planted.returncode == 0 and "planted mistake caught" in planted.stdout, planted.stdout + planted.stderr
