"""The engine's host code (dsm_engine.cpp: allocation, routes, launch shapes) built with g++
over a host-only stand-in for the HIP runtime and the kernel launchers
(tests/sanitize/fake_hip.cpp), under AddressSanitizer + UndefinedBehaviorSanitizer.  "Device"
memory is host memory, so a range too small or a pointer left null by a failed allocation
shows without a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SAN = os.path.join(ROOT, "tests", "sanitize")
CSRC = os.path.join(ROOT, "gpu_dsm_amd", "csrc")
HIP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(HIP, "hip")),
                                reason="g++ or the HIP headers not available")


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("engine") / "engine_checks")
    r = subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-fsanitize=address,undefined", "-fno-omit-frame-pointer",
                        "-fno-sanitize-recover=undefined", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
                        "-I", CSRC, "-I", HIP, os.path.join(CSRC, "dsm_engine.cpp"), os.path.join(SAN, "fake_hip.cpp"),
                        os.path.join(SAN, "engine_checks.cpp"), "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(which):
        p = subprocess.run([exe, which], capture_output=True, text=True, timeout=300,
                           env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1"))
        out = p.stdout + p.stderr
        assert p.returncode == 0 and "engine checks (%s): 0 failures" % which in out, out[-4000:]
    return run


def test_every_allocation_may_fail(checks):
    """Each device allocation of a session fails in turn, alone or with all that follow: the
    call is refused or done, the ensembles there are go on, and the repeated call succeeds."""
    checks("alloc")


def test_a_refused_ensemble_is_refused_again(checks):
    """A GEX background without quantiles, and a block factor that does not divide the lags."""
    checks("refused")


def test_lane_records_give_way(checks):
    """With the lane form's records in memory, any one failed allocation is made good by giving
    them back; without its tables or records a pass runs in the other forms."""
    checks("lanes")


def test_waves_per_cu_are_bounded_in_every_form(checks):
    checks("waves")


def test_concurrent_option_is_obeyed(checks):
    checks("concurrent")


@pytest.mark.parametrize("rule", ["lane", "share", "flow", "solo", "solo_flow", "bin2"])
def test_route(checks, rule):
    """The form a pass runs in, where the two sides of the rule were measured well apart."""
    checks("route_" + rule)


def test_window_parameters_need_no_pinned_memory(checks):
    checks("window")
