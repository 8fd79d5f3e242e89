"""The packed attention's scratch and work plan (csrc/sdq_sdpa_plan.h), swept on
the CPU: no launch of any call may need more than the call's scratch."""
import os
import subprocess

from conftest import PKG, ROOT


def test_every_launch_fits_its_scratch(tmp_path):
    exe = str(tmp_path / "sdpa_plan")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "sdpa_plan.cpp"), "-o", exe], check=True)
    env = {k: v for k, v in os.environ.items() if k != "SDQ_SDPA_SPLIT"}
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
