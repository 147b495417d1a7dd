"""gr_linear's choice of tile and the decoder's choice of gr_linear, without a GPU."""

import pytest

from vllm_gr_amd.v1.sid_decoder import _own_sizes


def _tile(lib, m, n, k, swiglu=0):
    t = lib.gr_linear_tile(m, n, k, swiglu)
    return t // 1000, t % 1000


def _rounds(m, rows, tile):
    """Rounds of workgroups, one to a CU, on the fullest of the 8 XCDs of 32 CUs: column tiles go round the XCDs whole."""
    return -(-(-(-(-(-rows // tile[1])) // 8) * -(-m // tile[0])) // 32)


@pytest.mark.parametrize("m,n,k,swiglu", [(448, 2160, 1408, 0), (188, 5376, 1408, 0), (277, 3136, 1920, 0),
                                          (415, 2192, 2048, 0), (430, 4608, 2048, 0), (334, 5376, 1664, 1)])
def test_tiles_fill_each_xcd_in_one_round(built_lib, m, n, k, swiglu):
    """These sizes have at most 256 of some smaller tile, but more than 32 of them on one XCD."""
    tile = _tile(built_lib, m, n, k, swiglu)
    assert _rounds(m, n * (1 + swiglu), tile) == 1


def test_tile_arguments(built_lib):
    assert built_lib.gr_linear_tile(0, 64, 512, 0) == built_lib.gr_linear_tile(4, 0, 512, 0) == 0
    assert _tile(built_lib, 1, 16, 512) == (64, 64)


@pytest.mark.parametrize("m,rows,k,swiglu", [(384, 4096, 2048, False), (368, 3072, 2048, False), (272, 6144, 2048, False),
                                             (512, 65536, 1024, False), (136, 32768, 2048, False), (64, 1024, 2048, False),
                                             (448, 2 * 14336, 2048, True), (640, 4096, 2048, False), (8, 2048, 6144, False)])
def test_sizes_where_the_library_measured_faster_stay_there(m, rows, k, swiglu):
    assert not _own_sizes(m, rows, k, swiglu)


@pytest.mark.parametrize("m", [1, 8, 100, 200, 512])
def test_decode_step_projections_are_own(m):
    """qkv, gate_up and lm_head of the 2048-feature decoder (o: but for 64 and 128 rows)."""
    for rows, swiglu in ((4096, False), (2048, False), (12288, True), (8192, False)):
        assert _own_sizes(m, rows, 2048, swiglu)
