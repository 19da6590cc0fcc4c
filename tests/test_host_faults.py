"""Failures that the host code has to survive, on the CPU: an allocation that
does not succeed, a call from another thread at a bad moment.  The scenarios are
in host_scenarios.py, their HIP runtime in native/fake_hip.cpp."""
import os
import subprocess
import sys

import pytest

import gsim

HERE = os.path.dirname(os.path.abspath(__file__))

SCENARIOS = ["failed_form_keeps_the_last", "lost_tree_buffers",
             "given_up_sort_is_never_read", "new_buffers_are_cleared_before_use",
             "query_beside_a_capture", "walk_form_by_the_members",
             "partial_sums_without_room_and_given_back",
             "knob_without_effect_keeps_the_graphs", "columns_asked_for_are_taken",
             "failed_requests_leave_their_space"]


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "native", "fake_hip.cpp")], check=True)
    return out


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_host_survives(fake_hip, scenario):
    gsim.load_library()  # built
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_scenarios.py"), fake_hip,
                        scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
