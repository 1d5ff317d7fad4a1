"""CPU checks of csrc/vb_staging.cpp (vb_get_phi's way through pinned memory):
tests/staging_check.cpp stands in for the HIP calls it makes; built with the
thread sanitizer."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("staging") / "check")
    csrc = os.path.join(ROOT, "cudabubble_amd", "csrc")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I" + csrc, "-o", exe, os.path.join(ROOT, "tests", "staging_check.cpp"),
                        os.path.join(csrc, "vb_staging.cpp"), "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("what", ["sizes", "threads", "pool", "launch_failure", "no_pinned", "make"])
def test_staging(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[-3000:]
