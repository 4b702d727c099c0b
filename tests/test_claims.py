"""How the wavefronts of the mixed batch's persistent launch share its tiles (csrc/claims.hpp), host build:
every tile is run once, and no wavefront keeps tiles that an idle one could run, also where another
launch leaves room for only some of the workgroups."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wgpu-sigops_amd", "csrc")
LONGEST = 112  # a tile's longest time in the schedule (100 .. 112)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("claims") / "libclaims.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I" + CSRC, "-o", so,
                    os.path.join(HERE, "devcheck", "claims_check.cpp")], check=True)
    L = ctypes.CDLL(so)
    L.tc_run.restype = ctypes.c_long
    L.tc_run.argtypes = [ctypes.c_uint32] * 4 + [ctypes.c_long, ctypes.c_uint32, ctypes.c_void_p]
    return L


# compute units, workgroups: one and two rounds of the MI355X's, a device with few compute units, and
# a grid that is no whole number of rounds (all tiles from the counter)
@pytest.mark.parametrize("cus,workgroups", [(256, 512), (256, 256), (4, 8), (0, 100)])
@pytest.mark.parametrize("room", [1.0, 0.5, 0.125])
def test_tiles_are_shared(lib, cus, workgroups, room):
    waves = 4 * workgroups
    rooms = max(1, int(room * workgroups))
    for ntiles in (0, 1, 63, 64, 65, waves // 2, waves - 1, waves, waves + 1, 2 * waves, 4 * waves, 4 * waves + 1):
        for until in (10**9, 150):  # the room stays as it is; it opens while the first tiles run
            done = np.zeros(max(ntiles, 1), np.uint32)
            end = lib.tc_run(ntiles, cus, workgroups, rooms, until, 0, done.ctypes.data)
            assert np.all(done[:ntiles] == 1), (ntiles, until)
            # Graham's bound for list schedules on the wavefronts there is always room for, and one tile
            # more: a workgroup without a tile of its own ends before others have started
            assert end <= LONGEST * (ntiles / (4 * rooms) + 2), (ntiles, until, end)


@pytest.mark.parametrize("share", [0.02, 0.25, 0.5])
def test_tiles_go_to_free_simds(lib, share):
    """tiles that fill at most half of the SIMDs are not run by wavefronts that share theirs with another
    launch's while others are free"""
    cus, workgroups = 256, 512
    ntiles = int(share * 4 * cus)
    done = np.zeros(ntiles, np.uint32)
    end = lib.tc_run(ntiles, cus, workgroups, workgroups, 0, 128, done.ctypes.data)
    assert np.all(done == 1) and end <= LONGEST, end
