"""What the host code launches, without a GPU.

tests/launch/launch_checks.cpp is linked with the library's objects and a HIP
runtime that runs no kernel and writes each launch down (fake_hip.cpp): refused
launches and allocations, the routes that sizes take, the arguments of launches.
"""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM", "/opt/rocm")
CSRC = os.path.join(ROOT, "grokking_abmod_amd", "csrc")
OBJECTS = os.path.join(ROOT, "grokking_abmod_amd", "_build")
HERE = os.path.join(ROOT, "tests", "launch")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                                reason="no host compiler or no HIP headers")


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    subprocess.run(["make", "-s", "-j", "8", "-C", CSRC], check=True)
    objects = [os.path.join(OBJECTS, f) for f in sorted(os.listdir(OBJECTS))
               if f.endswith(".o") and f not in ("capi.o", "mesh_gpt_cli.o", "mesh_gpt_bench.o")]
    exe = str(tmp_path_factory.mktemp("launch") / "launch_checks")
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                            "-I", CSRC, os.path.join(HERE, "launch_checks.cpp"), os.path.join(HERE, "fake_hip.cpp"),
                            *objects, "-o", exe], capture_output=True, text=True)
    assert built.returncode == 0, built.stderr
    return exe


@pytest.mark.parametrize("name", ["refused_launches", "foreign_errors", "window_launches", "window_routes", "chain_shapes",
                                  "scratch_limits", "chain_routes", "split_routes", "finite_checks",
                                  "no_batch", "threads_reading", "batch_without_memory",
                                  "wide_routes"])
def test_launches(checks, name):
    run = subprocess.run([checks, name], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout + run.stderr
