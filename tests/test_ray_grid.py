"""The ray indices of traversal launches (ray_grid.h, which also builds for the
host) up to 2^32 - 1 rays: every lane's rays are below n and none comes twice,
and a launch's threads fit 32 bits."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
WHOLE = 1 << 22  # kWholeGrid


@pytest.fixture(scope="module")
def grid_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("grid") / "grid_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", os.path.join(HERE, "grid_check.cpp"), "-o", exe])
    return exe


# a launch over all rays, and persistent grids
@pytest.mark.parametrize("limit", [WHOLE, 3072, 1])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 2073600, 2**30 - 1, 2**30 + 1, 2**31 - 1, 2**31, 2**31 + 12345,
                               4246732800, 2**32 - 257, 2**32 - 256, 2**32 - 255, 2**32 - 1])
def test_every_ray_once(grid_check, n, limit):
    for wave_rays in (64, 1) if n <= 2**24 else (64,):
        if limit == 1 and n > 2**24:
            continue  # millions of strides a lane
        threads_bad, places, rays, most = map(
            int, subprocess.check_output([grid_check, str(n), str(wave_rays), str(limit)]).split())
        assert not threads_bad and places == 0 and rays == 0
        if limit == WHOLE:
            assert most <= 4
