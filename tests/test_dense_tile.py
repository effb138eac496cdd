"""The rule by which a bf16 product takes its tile (cera_hip_dense_tile): plain arithmetic, checked without a GPU."""
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
