"""Rules of the engine's C++ interior that need no GPU, through a test-only host
library."""

import ctypes
import os
import subprocess

import pytest
import torch

from pysa_amd import _lib

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_probe")
INVALID_VALUE = 1  # hipErrorInvalidValue


@pytest.fixture(scope="module")
def probe():
    if torch.cuda.device_count():
        pytest.skip("a launcher that failed to refuse would launch")
    subprocess.run(["make", "-s", "-C", HERE], check=True)
    ctypes.CDLL(_lib.load()._name, mode=ctypes.RTLD_GLOBAL)
    return ctypes.CDLL(os.path.join(HERE, "_build", "libhost_probe.so"))


@pytest.fixture(scope="module")
def staging():
    subprocess.run(["make", "-s", "-C", HERE], check=True)
    lib = ctypes.CDLL(os.path.join(HERE, "_build", "libstaging_check.so"))
    lib.staging_without_pinned.argtypes = [ctypes.c_size_t]
    lib.staging_kept.argtypes = [ctypes.POINTER(ctypes.c_size_t), ctypes.c_int]
    lib.staging_kept.restype = lib.staging_alive.restype = ctypes.c_longlong
    return lib


# The schedule of the next sweep is written and read in one step below three
# blocks (block-random order); below two, steps are read that do not exist.
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("order,nblk", [(3, 1), (3, 2), (0, 1)])
@pytest.mark.parametrize("tiles", [1, 2])
def test_pipelined_launchers_refuse_short_schedules(probe, kind, order, nblk, tiles):
    assert probe.probe_launch_pipe(kind, order, nblk, tiles) == INVALID_VALUE


# (lanes a tile, reads' replicas): 64 lanes with whole reads from lane 0, or two
# batched tiles of 32 lanes; the lanes behind the last whole read are idle.
@pytest.mark.parametrize("tile", [32, 64])
def test_exchange_walk_reads_energies_inside_the_workgroup(probe, tile):
    for R in range(1, tile + 1):
        per = tile // R * R  # lanes of whole reads
        for lane in range(64):
            t, q = lane // tile * tile, lane % tile
            b0 = t + q // R * R
            # the last replica everywhere below but in idle lanes
            below = R - 1 if max(lane - 1, 0) % tile < per else 0
            got = probe.probe_lane_below(b0, below)
            assert 0 <= got < 64
            if q < per and lane > b0:
                assert got == b0 + below


# 8 KB, and just below, at and above what pinned memory takes
@pytest.mark.parametrize("bytes_", [1, 8192, (1 << 19) - 256, 1 << 19, (1 << 20) + 1])
def test_staging_without_pinned_memory_leaves_no_error(staging, bytes_):
    assert staging.staging_without_pinned(bytes_) == 0


def test_staging_keeps_little_memory(staging):
    mb = 1 << 20
    for sizes in ([1024], [mb, 1024], [1024, 7 * mb, 20 * mb, 100], [8 * mb, 8 * mb + 1]):
        kept = staging.staging_kept((ctypes.c_size_t * len(sizes))(*sizes), len(sizes))
        assert 0 < kept <= 32 * mb  # four arrays a call
        assert staging.staging_alive() == 0
