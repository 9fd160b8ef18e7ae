"""The library's workspaces (qengine_amd/csrc/workspace.cpp) on a host model of the HIP calls that they make
(workspace_host.cpp), linked by g++: one scenario per case. CPU only."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qengine_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ws") / "workspace_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    os.path.join(HERE, "workspace_host.cpp"), os.path.join(CSRC, "workspace.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["threads_on_one_stream", "another_stream_runs", "captures_have_their_own",
                                      "graphs_give_back", "allocate_beside_a_capture", "capture_without_memory", "growth_frees",
                                      "without_memory"])
def test_workspace(model, scenario):
    r = subprocess.run([model, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), r.stdout + r.stderr


@pytest.mark.parametrize("scenario,msg", [("reserve_in_capture", "called during graph capture"),
                                          ("reserve_without_memory", "no memory for 1048576 bytes")])
def test_reserve_that_cannot_be_met(model, scenario, msg):
    r = subprocess.run([model, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 3 and "FATAL" in r.stdout and msg in r.stderr, r.stdout + r.stderr
