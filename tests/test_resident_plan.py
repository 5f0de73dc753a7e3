"""The layout rule of the many-token product (llm_amd/csrc/resident_plan.h,
plain C++) on the CPU: tests/resident_plan_driver.cpp."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plans_cover_every_product_once(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = str(tmp_path / "plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(ROOT, "tests", "resident_plan_driver.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
