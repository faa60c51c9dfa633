"""Where the projections' shared tiles begin and end, and where the times that they were drawn by lie."""
import pytest

from chunk_attn import capi


# us on one GPU (MI355X) here, and the library's products (with the rotary launch for three weights), as measured
@pytest.mark.parametrize("rows,n_in,n_out,weights,pays", [
    (512, 4096, 4096, 3, True),          # 52.3 to 64, 86.4 to 96
    (2048, 4096, 4096, 3, True),         # 181 to 193 by machine, 209 to 212
    (2560, 4096, 4096, 3, False),        # 232.1, 230.0
    (4096, 2048, 2048, 3, True),         # 101.2, 120.1
    (8192, 1024, 1024, 3, True),         # 63.8, 81.0
    (1600, 5120, 5120, 3, False),        # 269.1, 270.8
    (1000, 4096, 4096, 1, True),         # 33.6, 40.1
    (2048, 4096, 4096, 1, True),         # 58.5, 63.3
    (2300, 4096, 4096, 1, False),        # 87.5, 69.5
    (4096, 2048, 2048, 1, True),         # 32.2, 37.3
    (6000, 2048, 2048, 1, False),        # 53.0, 46.9
    (8192, 1024, 1024, 1, True),         # 19.7, 24.0
    (16000, 1024, 1024, 1, False),       # 37.4, 31.9
    (64, 8192, 8192, 3, False),          # weights past what was measured
])
def test_shared_tiles_are_taken_where_they_are_faster(rows, n_in, n_out, weights, pays):
    assert capi.shared_tiles_pay(rows, n_in, n_out, weights) == pays


@pytest.mark.parametrize("n,tile", [(4096, 256), (1000, 256), (256, 256), (255, 256)])
def test_shared_tiles_stop_behind_whole_rounds(n, tile):
    """One weight: while the tiles of 128 x 256 fit 256 compute units at once; three: up to three rounds of them."""
    columns = -(-n // tile)
    for weights, tiles in ((1, 256), (3, 768)):
        rows = tiles // (columns * weights) * 128
        assert capi.shared_tiles_pay(rows, n, n, weights) and not capi.shared_tiles_pay(rows + 1, n, n, weights)
