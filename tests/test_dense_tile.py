"""The rules by which a bf16 product takes its tile (cera_hip_dense_tile, cera_hip_dense_streams_tile): plain arithmetic, checked without a GPU."""
import subprocess
from pathlib import Path

import pytest

from cera_amd import hip_api

N_CU, XCDS = 256, 8


def _rounds(rows, n):
    """Rounds of one 256 x 256 workgroup per CU on the XCD that gets most of them: a weight tile's workgroups all go to the
    XCD of its index modulo eight."""
    most = max(len(range(x, -(-rows // 256), XCDS)) for x in range(XCDS)) * -(-n // 256)
    return -(-most // (N_CU // XCDS))


@pytest.mark.parametrize("rows,k,n,tile", [(28672, 4096, 512, 256), (5120, 3072, 2048, 256), (17920, 2560, 640, 256),
                                           (21504, 3072, 640, 128), (21504, 3072, 513, 128), (10752, 3072, 1300, 128),
                                           (3072, 3072, 2048, 128), (4096, 18432, 1900, 128), (36864, 4096, 128, 128), (28672, 4096, 128, 64)])
def test_tiles(rows, k, n, tile):
    assert hip_api.dense_tile(rows, k, n) == tile


def test_the_largest_tiles_fill_their_rounds():
    """At least 55 % of what the chip computes in the rounds of its fullest XCD, counted one workgroup at a time."""
    seen = set()
    for rows in range(256, 40000, 1280):
        for n in range(129, 2100, 123):
            fills = rows * n / (_rounds(rows, n) * N_CU * 256 * 256)
            got = hip_api.dense_tile(rows, 4096, n) == 256
            assert got == (fills >= 0.55), (rows, n, fills)
            seen.add(got)
    assert seen == {True, False}


@pytest.mark.parametrize("rows,k,n,streams,want", [(3072, 1030, 2040, 4, (256, 2)), (3000, 1100, 2047, 3, (256, 2)), (3072, 8200, 1010, 4, (256, 3)),
                                                   (4096, 8300, 600, 2, (256, 4)), (3072, 64, 2048, 4, (128, 1)), (2048, 8192, 2048, 4, (128, 2)),
                                                   (5200, 200, 1800, 4, (256, 1)), (2048, 2048, 40, 4, (64, 8)), (2048, 2048, 40, 3, (64, 8))])
def test_tiles_of_streams(rows, k, n, streams, want):
    assert hip_api.dense_streams_tile(rows, k, n, streams) == want


@pytest.mark.parametrize("streams", [1, 3, 4])
def test_streams_with_less_room_take_the_next_smaller_plan(streams):
    """Two parts on 256 x 256 tiles; with room for one part's sums the 128 x 128 tiles, as if there were no larger ones; without, K whole,
    four streams by small tiles."""
    rows, k, n = 3072, 1030, 2048
    one = rows * n * 4
    for room, want in ((2 * one, (256, 2)), (2 * one - 1, (128, 1)), (one, (128, 1)), (one - 1, (64 if streams == 4 else 128, 1)), (0, (64 if streams == 4 else 128, 1))):
        assert hip_api.dense_streams_tile(rows, k, n, streams, room) == want


@pytest.mark.parametrize("rows,k,n,want", [(4096, 18400, 1900, (256, 2)), (3072, 11264, 700, (256, 5)), (6144, 4090, 1400, (256, 1)), (5120, 8192, 1400, (128, 1)),
                                           (4096, 4096, 1900, (128, 1)), (3072, 2048, 1568, (128, 2)), (4096, 18432, 130, (128, 8)), (8192, 1984, 1000, (128, 1))])
def test_larger_tiles_in_parts_of_k(rows, k, n, want):
    """Products that with K whole would take 128 x 128 tiles: 256 x 256 ones in the parts that are estimated fastest, where they are by far;
    from 2048 columns and 129 tokens on."""
    assert hip_api.dense_tile(rows, k, n) == 128
    assert hip_api.dense_streams_tile(rows, k, n, 0) == want


def test_less_room_takes_the_smaller_tiles():
    rows, k, n = 4096, 18432, 2000
    assert hip_api.dense_streams_tile(rows, k, n, 0, 2 * rows * n * 4) == (256, 2)
    assert hip_api.dense_streams_tile(rows, k, n, 0, 2 * rows * n * 4 - 1) == (128, 1)


@pytest.mark.parametrize("rows,k,n,want", [(3072, 8192, 690, (256, 5)), (4096, 14336, 520, (256, 5)), (2048, 8192, 850, (256, 8)), (3072, 8192, 1450, (256, 2)),
                                           (3072, 1984, 1450, (128, 2)), (2048, 8192, 400, (128, 8))])
def test_streams_in_more_parts_of_k(rows, k, n, want):
    """Where two to four parts do not fill their rounds, as without streams."""
    assert hip_api.dense_streams_tile(rows, k, n, 4) == want


def test_the_plan_and_its_workspace_agree(tmp_path):
    """No product asks for a workspace that its plan does not use, and none has a plan whose sums it was refused."""
    root = Path(__file__).resolve().parent.parent
    exe = tmp_path / "dense_plan_room"
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{root / 'cera_amd' / 'csrc'}", str(root / "tests" / "native" / "dense_plan_room.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert " 0 of them" not in r.stdout
