"""Host code of the library on a runtime without a GPU (tests/abi/fake_hip.hpp): what calls do when allocations or
launches fail, and what they share between threads."""
import os
import subprocess

import pytest

import hopefoam_amd.dgh as dgh

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIBDIR = os.path.dirname(dgh.lib_path())


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    out = str(tmp_path_factory.mktemp("host") / "host_paths")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "hopefoam_amd", "csrc"), "-isystem", os.path.join(rocm, "include"),
                    os.path.join(HERE, "abi", "host_paths.cpp"), "-o", out, "-L" + LIBDIR, "-ldghip",
                    "-Wl,-rpath," + LIBDIR, "-L" + os.path.join(rocm, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + os.path.join(rocm, "lib"), "-lpthread"], check=True)
    return out


def run(program, name):
    p = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout == "ok\n", p.stderr


def test_error_is_not_kept(program):
    """an allocation that fails is an error of its own call only"""
    run(program, "error_is_not_kept")


@pytest.mark.parametrize("name", ["lserk4_scratch", "ssprk2_scratch"])
def test_failing_scratch(program, name):
    """a time loop whose scratch fields cannot be allocated fails, and the next call finds them allocated"""
    run(program, name)


def test_sipg_rhs_threads(program):
    """right-hand sides of one solver formed by two threads at once keep their boundary data apart"""
    run(program, "sipg_rhs_threads")


def test_ensemble_failing_launch(program):
    """an ensemble call that fails half-way leaves nothing running"""
    run(program, "ensemble_failing_launch")


def test_ensemble_failing_shape(program):
    """a tile shape that cannot be taken for want of memory leaves the ensemble's work list and shapes as they were"""
    run(program, "ensemble_failing_shape")


def test_staging_as_needed(program):
    """a context takes as much pinned memory as its transfers need"""
    run(program, "staging_as_needed")
