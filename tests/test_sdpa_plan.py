"""The packed attention's scratch and work plan (csrc/sdq_sdpa_plan.h), swept on
the CPU: no launch of any call may need more than the call's scratch, nor that
more than its bound, also with a forced number of shares."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "sdpa_plan")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "sdpa_plan.cpp"), "-o", exe], check=True)

    def run(split, *args):
        env = {k: v for k, v in os.environ.items() if k != "SDQ_SDPA_SPLIT"}
        if split is not None:
            env["SDQ_SDPA_SPLIT"] = split
        return subprocess.run([exe, *args], capture_output=True, text=True, timeout=120, env=env)

    return run


@pytest.mark.parametrize("split", [None, "1", "3", "16"])
def test_every_launch_fits_its_scratch(plan, split):
    r = plan(split)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("split,cut", [("0", (1, 24)), ("1", (1, 24)), ("3", (3, 8)),
                                       ("5", (5, 5)), ("16", (12, 2)), ("99", (12, 2))])
def test_forced_shares(plan, split, cut):
    """SDQ_SDPA_SPLIT: a factor from 2 to 16, no cut below."""
    assert plan(split, "cut").stdout == "%d shares of %d blocks\n" % cut
