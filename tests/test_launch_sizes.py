"""The lanes per slot of a lane-group launch (pbf_types.h, launch_lanes): as many as asked for while the launch's
work items stay below 2^32, at most half as many above, for every scene a solver accepts (2^28 slots)."""
import os
import subprocess

import pytest

from conftest import ROOT

SLOTS = [1, 255, 1 << 18, (1 << 27) - 2049, 1 << 27, (1 << 28) - 2049, (1 << 28) - 2048, (1 << 28) - 1, 1 << 28]


@pytest.fixture(scope="module")
def lanes_of(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    src = d / "lanes.cpp"
    src.write_text('#include "pbf_types.h"\n#include <cstdio>\n#include <cstdlib>\n'
                   'int main(int c, char** v) { for (int k = 1; k + 1 < c; k += 2) std::printf("%d\\n", '
                   'akua::launch_lanes((uint32_t)std::strtoul(v[k], nullptr, 10), std::atoi(v[k + 1]))); }\n')
    exe = d / "lanes"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__=1", f"-I{rocm}/include",
                    f"-I{ROOT}/akuaengine_amd/csrc", str(src), "-o", str(exe)], check=True)
    return lambda pairs: [int(x) for x in subprocess.run([str(exe), *[str(v) for p in pairs for v in p]], check=True,
                                                         capture_output=True, text=True).stdout.split()]


def test_work_items_stay_below_2_to_the_32(lanes_of):
    pairs = [(n, lanes) for n in SLOTS for lanes in (1, 2, 4, 8, 16)]
    for (n, lanes), got in zip(pairs, lanes_of(pairs)):
        rounded = -(-n // 2048) * 2048  # workgroups of 256 work items, a multiple of eight of them
        assert rounded * got < 1 << 32
        assert got == lanes or 2 * got * (n + 2048) >= 1 << 32
        if n <= 1 << 27:
            assert got == lanes
