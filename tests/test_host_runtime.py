"""The library's host code (flip_api.cpp, hash_api.cpp, unet_api.cpp) over a stand-in for the HIP runtime
that queues work until something waits for it and can run out of memory or fail a launch
(host/fake_hip.hpp): what happens between calls, without a GPU."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "aquarius_amd" / "csrc"
HOST = ROOT / "tests" / "host"


@pytest.fixture(scope="module")
def host_cases(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host") / "host_cases"
    subprocess.run(["/opt/rocm/bin/amdclang++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-D__align__(n)=__attribute__((aligned(n)))", "-DHIP_SYMBOL(x)=(const void*)(x)", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    f"-I{CSRC}", str(HOST / "host_cases.cpp"), str(CSRC / "flip_api.cpp"), str(CSRC / "flip_seed.cpp"),
                    str(CSRC / "hash_api.cpp"), str(CSRC / "unet_api.cpp"), "-o", str(exe), "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("name", [
    "four_phases_on_small_grids",
    "paired_tiles_by_fluid",
    "sparse_particles_on_small_grids",
    "one_workgroup_per_tile",
    "tiles_fit_the_grid",
    "exports_need_little_memory",
    "sort_by_density",
    "network_after_failed_growth",
    "kept_blocks_stay_on_their_device",
    "kept_memory_is_given_back",
    "eight_chunk_lengths_replay",
    "timed_small_steps",
    "replayed_step_marks_content",
    "iterate_after_a_failed_capture",
    "mgpcg_after_a_failed_solve",
    "solves_after_a_failed_launch",
    "solve_returns_idle",
    "hash_after_failed_growth",
    "hash_after_a_failed_sort",
    "load_after_clear",
])
def test_host(host_cases, tmp_path, name):
    r = subprocess.run([str(host_cases), name, str(tmp_path)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
