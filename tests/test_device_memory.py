"""The device memory bookkeeping of the library's host code, on the CPU against
a stand-in device (arena_main.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.environ.get("ROCM_PATH", "/opt/rocm") + "/include"


@pytest.fixture(scope="module")
def arena_main(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.exists(os.path.join(HIP, "hip", "hip_runtime.h")):
        pytest.skip("no g++ or HIP headers")
    exe = tmp_path_factory.mktemp("arena") / "arena_main"
    csrc = os.path.join(ROOT, "gds2para_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-w", "-D__HIP_PLATFORM_AMD__", "-I", HIP, "-I", csrc, "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "arena_main.cpp"),
                    os.path.join(csrc, "status.cpp"), "-o", str(exe)], check=True)
    return exe


def _run(exe, scenario):
    r = subprocess.run([str(exe), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_failed_setup_frees_its_temporaries(arena_main):
    """A setup step that leaves early gives back every temporary, the pool's and
    those allocated by themselves."""
    _run(arena_main, "failed_setup")


def test_idle_chunks_are_given_back_when_memory_runs_out(arena_main):
    """The pool's idle chunks never make an allocation fail that would succeed
    without them."""
    _run(arena_main, "idle_chunks")


def test_pool_buffers(arena_main):
    """Buffers of a scope lie apart and inside what the device gave, and all of
    it is given back."""
    _run(arena_main, "pool")


def test_arena_counts_what_it_holds(arena_main):
    """An arena's byte counter (what gp_layout_device_bytes adds up) is the
    memory it holds of the device, slabs whole and released buffers included
    while their slab stays."""
    _run(arena_main, "bytes")


def test_counting_arena_matches_an_allocating_one(arena_main):
    """The sizes of gp_solve_workspace_bytes come from the allocation code run
    on arenas that only count."""
    _run(arena_main, "count_only")
