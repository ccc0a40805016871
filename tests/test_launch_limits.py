"""The z chunks of a launch that lays all its blocks along one axis
(sw_launch.hpp): the asked length wherever that fits, and never more than 2^32-1
threads, also on grids of few points along y that fill the device's memory."""
import os
import shutil
import subprocess

import harness

CSRC = os.path.join(harness.REPO, "simwave_amd", "csrc")
SOURCE = r"""
#include <cstdio>
#include "sw_launch.hpp"
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
int main()
{
    // 384^3 and 2000^3 points, interior rows of 8 lines and 64 points
    CHECK(sw::z_chunk_planes(8, 6 * 48, 384, 512, 1000) == 8);
    CHECK(sw::z_chunk_planes(8, 32 * 250, 2000, 512, 1000) == 8);
    // 50000 x 50000 x 4 points of radius 1: 39 M blocks of 8 planes
    const long long cols = (50000 - 2 + 7) / 8;
    const int p = sw::z_chunk_planes(8, cols, 49998, 512, 1000);
    CHECK(!sw::launch_fits(cols * ((49998 + 7) / 8), 512));
    CHECK(p == 64 && sw::launch_fits(cols * ((49998 + p - 1) / p) + 1000, 512));
    CHECK(sw::z_chunk_planes(1, 8388607, 5, 512, 0) == 5);
    CHECK(sw::z_chunk_planes(1, 8388607, 1, 512, 0) == 1);
    CHECK(sw::z_chunk_planes(256, 1 << 20, 100, 512, 0) == 256);
    CHECK(sw::launch_fits(8388607, 512) && !sw::launch_fits(8388608, 512));
    for (long long c = 1; c < 8000000; c = c * 3 + 1)
        for (int iz = 1; iz < 3000000; iz = iz * 5 + 2) {
            const int q = sw::z_chunk_planes(8, c, iz, 512, 4096);
            CHECK(q >= 8 || q == iz);
            CHECK(sw::launch_fits(c * ((iz + q - 1) / q) + 4096, 512));
            CHECK(q == 8 || !sw::launch_fits(c * ((iz + 7) / 8) + 4096, 512));
        }
    printf("ok\n");
    return 0;
}
"""


def test_z_chunks_fit_one_launch(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    src, exe = tmp_path / "launch.cpp", tmp_path / "launch"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.stdout == "ok\n" and res.returncode == 0, res.stdout
