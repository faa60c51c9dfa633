"""Where the projections' shared tiles begin and end, and where the times that they were drawn by lie."""
import ctypes

import pytest

from chunk_attn import capi
import test_gpu_shared_tiles as gpu


# us on one GPU (MI355X) here, and the library's products (with the rotary launch for three weights), as measured on
# weights from memory
@pytest.mark.parametrize("rows,n_in,n_out,weights,pays", [
    (512, 4096, 4096, 3, True),          # 67, 110
    (2048, 4096, 4096, 3, True),         # 180, 234
    (2560, 4096, 4096, 3, False),        # 254, 251
    (4096, 2048, 2048, 3, True),         # 96, 131
    (8192, 1024, 1024, 3, True),         # 55, 85
    (1600, 5120, 5120, 3, False),        # 288 to 301, 307
    (1000, 4096, 4096, 1, True),         # 38, 42
    (2048, 4096, 4096, 1, True),         # 66, 72
    (2300, 4096, 4096, 1, False),        # 98, 74
    (4096, 2048, 2048, 1, True),         # 36, 39
    (6000, 2048, 2048, 1, False),        # 59, 50
    (8192, 1024, 1024, 1, True),         # 24, 26
    (16000, 1024, 1024, 1, False),       # 42, 35
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


def tile(rows, n_out, n_in, rotary):
    r, c = ctypes.c_int(), ctypes.c_int()
    capi._check(capi.load().ca_projection_tile(rows, n_out, n_in, rotary, r, c))
    return r.value, c.value


def sizes(test):
    (mark,) = [m for m in test.pytestmark if m.name == "parametrize"]
    return mark.args[1]


def test_the_gpu_tests_of_the_tiles_of_three_heads_reach_them():
    found = [tile(rows, heads * 128, n_in, 1) for rows, heads, n_in in sizes(gpu.test_qkv_rotary_in_tiles_of_three_heads)]
    assert found == [(128, 384)] * 4 + [(256, 384)] * 3


def test_the_gpu_tests_of_shared_tiles_reach_every_one():
    plain = {tile(rows, n_out, n_in, 0) for rows, n_out, n_in in sizes(gpu.test_linear_in_shared_tiles)}
    assert plain == {(64, 64), (64, 128), (128, 128), (128, 256)}
    assert all(tile(300, 2050, n_in, 0) == (64, 64) for n_in in sizes(gpu.test_linear_in_the_smallest_shared_tiles))
    rotary = {tile(rows, heads * 128, n_in, 1) for rows, heads, n_in in sizes(gpu.test_qkv_rotary_in_shared_tiles)}
    assert rotary == {(64, 64), (64, 128), (128, 128), (128, 256)}


def test_residuals_reach_the_larger_tiles():
    """The prompts of test_native_model_pass_keeps_every_bit whose output projections add to the residual."""
    assert [tile(rows, hidden, hidden, 0) for rows, hidden in ((449, 1024), (660, 1536), (1100, 1024), (2000, 1536), (3001, 1024), (2100, 2048))] == [
        (64, 64), (64, 128), (64, 128), (128, 128), (128, 128), (128, 256)]


def test_tiles_of_a_size_that_is_none_are_refused():
    r = ctypes.c_int()
    for bad in ((0, 128, 64, 0), (1, 0, 64, 0), (1, 128, 63, 0), (1, 100, 64, 1)):
        assert capi.load().ca_projection_tile(*bad, r, r) == -1
    assert tile(1, 8, 64, 0) == tile(16, 8, 64, 0) == (16, 16) and tile(17, 8, 64, 0) == (32, 32)
