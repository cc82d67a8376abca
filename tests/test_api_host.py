"""CPU tests of the C ABI's host side (q-pso_amd/csrc/qpso_api.cpp) against a
mock HIP runtime (tests/api_mock.cpp): what the calls do when a copy cannot be
enqueued or there is no pinned memory, which calls allocate, and what a
solve's memory amounts to.  Built with AddressSanitizer and
UndefinedBehaviorSanitizer; the runtime itself is not linked."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
INC = ["-I", os.path.join(ROCM, "include"), "-I", os.path.join(REPO, "include"),
       "-I", os.path.join(REPO, "q-pso_amd", "csrc")]
FLAGS = ["-std=c++17", "-O1", "-g", "-ffp-contract=off", "-fwrapv", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__", "-fno-omit-frame-pointer",
         "-fsanitize=address,undefined", "-fno-sanitize-recover=all"]

SCENARIOS = ["results_wait_on_failure", "no_pinned_memory", "staging_keeps_its_size", "many_results",
             "arena_bytes"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("api"))
    out = os.path.join(d, "api_mock")
    subprocess.check_call(["g++", *FLAGS, *INC, "-o", out, os.path.join(REPO, "q-pso_amd", "csrc", "qpso_api.cpp"),
                           os.path.join(REPO, "tests", "api_mock.cpp"), "-lpthread"])
    return out


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_api_scenario(exe, scenario):
    p = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and f"PASS {scenario}" in p.stdout, p.stdout + p.stderr
