"""Where the projections' shared tiles begin and end, with the times on both sides of the lines."""
import pytest

from chunk_attn import capi


# us on one GPU (MI355X): here, and the library's products (with the rotary launch for three weights)
@pytest.mark.parametrize("rows,n_in,n_out,weights,here,library,pays", [
    (512, 4096, 4096, 3, 52.3, 86.4, True), (2048, 4096, 4096, 3, 180.5, 202.2, True), (2560, 4096, 4096, 3, 232.1, 230.0, False),
    (4096, 2048, 2048, 3, 101.2, 120.1, True), (8192, 1024, 1024, 3, 63.8, 81.0, True), (1600, 5120, 5120, 3, 269.1, 270.8, False),
    (1000, 4096, 4096, 1, 33.6, 40.1, True), (2048, 4096, 4096, 1, 58.5, 63.3, True), (2300, 4096, 4096, 1, 87.5, 69.5, False),
    (4096, 2048, 2048, 1, 32.2, 37.3, True), (6000, 2048, 2048, 1, 53.0, 46.9, False), (8192, 1024, 1024, 1, 19.7, 24.0, True),
    (16000, 1024, 1024, 1, 37.4, 31.9, False), (64, 8192, 8192, 3, 0, 0, False)])
def test_shared_tiles_are_taken_where_they_are_faster(rows, n_in, n_out, weights, here, library, pays):
    assert capi.shared_tiles_pay(rows, n_in, n_out, weights) == pays
    assert here <= library if pays else here >= library - 2
